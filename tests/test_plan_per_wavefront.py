"""The scheduler of the plan-per-wavefront kernel at the sizes where it changes form: one or two nodes to a lane
(64 / 65 lowered nodes), waiting nodes only (128 / 129), graphs whose waiting nodes outgrow the lanes (more than
60), the largest graph the kernel takes (384).  The host build of the same arithmetic schedules with an ordered
list, one pop per iteration; makespan, peak, score, mask and critical-chain mass are its bits, the utilisation is
that of the single-plan trace."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


@pytest.mark.parametrize("c,K", [(1, 3), (1, 5), (1, 10), (2, 6), (2, 16), (3, 3), (3, 6), (3, 10), (4, 1), (4, 16),
                                 (4, 58), (4, 59), (4, 64)])
def test_every_form_of_the_scheduler_equals_the_host_build(c, K):
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, 600)
    p = replace(cfg.problem, K_eval=K)
    want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16, want_mass=True)
    eng = Engine(p)
    eng.set_state_lanes(1)
    try:
        mass, util, plain = eng.eval_mass(batch, gate_stale=True), eng.eval_util(batch, gate_stale=True), eng.eval(batch, gate_stale=True)
        for out in (mass, util, plain):
            assert np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want[k]), k
        assert same_bits(mass["mass"], want["mass"])
        for i in np.flatnonzero((want["mask"] & abi.MASK_VALID) != 0)[::97]:
            assert float(util["util"][i]).hex() == float(eng.trace_metrics(batch, int(i))[0]).hex(), i
    finally:
        eng.close()


@pytest.mark.parametrize("c,K", [(1, 4), (3, 10), (1, 16)])
def test_one_plan_at_a_time_equals_the_oracle_on_either_side_of_the_largest_graph(c, K):
    """evaluate_cached and its trace: from one launch up to 384 nodes, over the staged path and the single-plan trace
    beyond (config 1 at 16 unrolled steps has graphs on either side)."""
    from oracle import rpeg_oracle as oracle
    from rpeg_amd.search.cache import EvalCache
    from rpeg_amd.search.evaluate import Configuration, evaluate_cached
    cfg, batch = seeded_batch(c, 3)
    p = cfg.problem
    for i in range(3):
        rpeg, plan, wl = batch.configuration(p, i)
        want = oracle.evaluate_plan(rpeg, plan, p.device_space, p.suite, wl, p.hw, K, p.memory_policy, check_stale=True,
                                    want_trace=True)
        score, trace, feasible, miss = evaluate_cached(Configuration(rpeg, plan, p.device_space), EvalCache(), p.suite, wl, p.hw, K)
        assert miss and score == want["score"] and feasible == want["feasible"]
        assert {n.id: t for n, t in trace.finish.items()} == want["finish"]
        assert list(trace.start) == list(trace.finish) and len(trace.start) == len(want["nodes"])
