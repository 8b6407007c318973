"""Threads that share an engine, as those do that evaluate plans of one problem through rpeg_amd.search: its calls are taken one at
a time."""

import dataclasses
import inspect
import threading
import time

import numpy as np
import pytest

from rpeg_amd import configs
from rpeg_amd.engine import abi
from rpeg_amd.engine.runtime import Engine
from rpeg_amd.search import candidates
from rpeg_amd.search.evaluate import Configuration, evaluate, evaluate_batch


def in_threads(calls):
    failed = []

    def run(call):
        try:
            call()
        except Exception as e:      # noqa: BLE001
            failed.append(e)
    threads = [threading.Thread(target=run, args=(call,)) for call in calls]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


def test_calls_of_two_threads_do_not_meet_in_the_library():
    inside, met = [], []

    class Library:
        def __getattr__(self, name):
            def call(*args):
                inside.append(name)
                met.append(len(inside))
                time.sleep(0.05)
                inside.pop()
                return 0
            return call

    eng = Engine.__new__(Engine)
    eng.lib, eng._h, eng._calls = Library(), None, threading.RLock()
    params = abi.SaParamsT()
    in_threads([lambda: eng.set_split_model(np.zeros(9)), lambda: eng.set_sa_groups(2), eng.stats, eng.host_us,
                lambda: eng.sa_propose(params, [], 1)])
    assert len(met) == 5 and max(met) == 1


def test_every_public_call_of_an_engine_is_one_of_these():
    for name, call in vars(Engine).items():
        if inspect.isfunction(call) and not name.startswith("_"):
            assert hasattr(call, "__wrapped__"), name


@pytest.mark.gpu
def test_threads_that_evaluate_plans_of_one_problem():
    cfg = configs.config(5)
    p = dataclasses.replace(cfg.problem, structures=cfg.problem.structures[:1])
    batch = candidates.generate(p, 240, cfg.tau_choices, seed=5, tag=5)
    plans = [Configuration(*batch.configuration(p, i)[:2], p.device_space) for i in range(batch.n)]
    alone = evaluate_batch(plans, p.suite, p.workload, p.hw, p.K_eval)
    single = [evaluate(c, p.suite, p.workload, p.hw, p.K_eval)[0] for c in plans[:8]]

    def part(k):
        for n in (7, 60, 1 + k):
            for at in range(30 * k, 240, 60):
                r = evaluate_batch(plans[at:at + n], p.suite, p.workload, p.hw, p.K_eval)
                for name in ("score", "makespan", "peak", "mask"):
                    assert np.array_equal(getattr(r, name), getattr(alone, name)[at:at + n]), (name, at, n)
            assert evaluate(plans[k], p.suite, p.workload, p.hw, p.K_eval)[0] == single[k]
    in_threads([lambda k=k: part(k) for k in range(4)])
