"""The text of a plan's cache key put together from its row of numbers, and plans packed many at a time, against the plain forms."""

import dataclasses
import threading
import time

import numpy as np
import pytest

from rpeg_amd import configs
from rpeg_amd.engine.problem import PlanBatch
from rpeg_amd.search import candidates, evaluate
from rpeg_amd.search.cache import _config_hash_plain, config_hash, key_text
from rpeg_amd.search.evaluate import Configuration, _pack, _structure_of
from rpeg_amd.search.optimizer import plan_row


def seeded(workload, structure, n):
    cfg = configs.config(workload)
    p = dataclasses.replace(cfg.problem, structures=cfg.problem.structures[structure:structure + 1])
    batch = candidates.generate(p, n, cfg.tau_choices, seed=3, tag=workload)
    return p, [batch.configuration(p, i)[:2] for i in range(n)]


CASES = [(1, 0), (2, 0), (3, 0), (3, 1), (4, 0), (5, 0)]


@pytest.mark.parametrize("workload,structure", CASES)
def test_key_of_a_row_is_the_key_of_its_plan(workload, structure):
    for rpeg, plan in seeded(workload, structure, 20)[1]:
        want = _config_hash_plain(rpeg, plan)
        assert config_hash(rpeg, plan) == want
        assert key_text(rpeg).of_row(plan_row(rpeg, plan).tolist()) == want


def test_plans_that_are_no_row_of_whole_numbers():
    _, [(rpeg, plan)] = seeded(1, 0, 1)
    v, w = rpeg.vertices[:2]
    other = dataclasses.replace(v, id="x%d")
    forms = [dataclasses.replace(plan, mb={**plan.mb, v: True}), dataclasses.replace(plan, mb={**plan.mb, v: 2.0}),
             dataclasses.replace(plan, pi={**plan.pi, v: (1, 2)}), dataclasses.replace(plan, pi={**plan.pi, v: [2, 1, 1]}),
             dataclasses.replace(plan, mb={x: m for x, m in plan.mb.items() if x != w}),
             dataclasses.replace(plan, sigma={**plan.sigma, other: plan.sigma[v]}),
             dataclasses.replace(plan, mb={**{x: m for x, m in plan.mb.items() if x != w}, other: 1}),
             dataclasses.replace(plan, sigma=dict(reversed(plan.sigma.items())))]
    for p in forms:
        assert config_hash(rpeg, p) == _config_hash_plain(rpeg, p)
    with pytest.raises(TypeError):      # (as json refuses it)
        config_hash(rpeg, dataclasses.replace(plan, mb={**plan.mb, v: np.int64(2)}))
    odd = dataclasses.replace(rpeg, vertices=(other,) + rpeg.vertices[1:])      # a name with a format character
    move = lambda d: {other if x == v else x: y for x, y in d.items()}  # noqa: E731
    p = dataclasses.replace(plan, sigma=move(plan.sigma), pi=move(plan.pi), mb=move(plan.mb))
    assert config_hash(odd, p) == _config_hash_plain(odd, p)


def test_a_key_makes_no_encoder(monkeypatch):
    """... neither a new template's nor that of a plan that is no row (six to ten a key were a tenth of its time)."""
    import json
    _, [(rpeg, plan), (other, _)] = seeded(1, 0, 2)
    half = dataclasses.replace(plan, mb={v: float(m) for v, m in plan.mb.items()})
    want = [_config_hash_plain(rpeg, plan), _config_hash_plain(other, half)]
    monkeypatch.setattr(json, "JSONEncoder", None)
    assert [config_hash(rpeg, plan), config_hash(other, half)] == want


@pytest.mark.parametrize("names", [(), (0, 1, 2, 3, 4, 5), (10, 9, 8, 7, 6, 5), (1.5, 2, True, 4, 5, 6), ("a",)])
def test_key_of_a_template_without_vertices_or_with_other_names_than_texts(names):
    _, [(rpeg, plan)] = seeded(1, 0, 1)
    verts = tuple(dataclasses.replace(v, id=x) for v, x in zip(rpeg.vertices, names))
    move = lambda d: dict(zip(verts, d.values()))  # noqa: E731
    for edges in ((), tuple(dataclasses.replace(e, src=verts[0], dst=verts[-1]) for e in rpeg.data_edges[:1] if verts)):
        r = dataclasses.replace(rpeg, vertices=verts, data_edges=edges, pub_edges=())
        p = dataclasses.replace(plan, sigma=move(plan.sigma), pi=move(plan.pi), mb=move(plan.mb))
        assert config_hash(r, p) == config_hash(r, p) == _config_hash_plain(r, p)


@pytest.mark.parametrize("workload,structure", CASES)
def test_packed_plans_are_the_plans_one_by_one(workload, structure):
    problem, plans = seeded(workload, structure, 9)
    st = _structure_of(plans[0][0])
    got = _pack([Configuration(r, p, problem.device_space) for r, p in plans], st, problem.workload)
    want = PlanBatch.empty(len(plans))
    for i, (r, p) in enumerate(plans):
        want.set_plan(i, 0, 1 if problem.workload.gen_quantiles else 0, [int(r.tau[m]) for m in st.tau_models], r, p)
    assert np.array_equal(got.vert, want.vert) and np.array_equal(got.head, want.head)
    assert got.vert.dtype == want.vert.dtype and got.head.dtype == want.head.dtype and got.vert.flags.c_contiguous


def test_plans_that_cannot_be_packed():
    problem, [(rpeg, plan)] = seeded(5, 0, 1)
    st, v = _structure_of(rpeg), rpeg.vertices[3]
    without = lambda d: {x: y for x, y in d.items() if x != v}  # noqa: E731
    for change, error in (({"sigma": without(plan.sigma)}, KeyError), ({"pi": without(plan.pi)}, KeyError),
                          ({"mb": without(plan.mb)}, KeyError), ({"pi": {**plan.pi, v: (1, 1)}}, ValueError),
                          ({"mb": {**plan.mb, v: 1 << 15}}, OverflowError),
                          ({"mb": {**plan.mb, v: 1 << 15, rpeg.vertices[0]: 2.0}}, OverflowError)):
        with pytest.raises(error):
            _pack([Configuration(rpeg, dataclasses.replace(plan, **change), problem.device_space)], st, problem.workload)


def test_an_engine_used_last_is_that_of_its_key(monkeypatch):
    """... also where another thread adds one between the comparison and the return."""
    problem, [(rpeg, plan)] = seeded(5, 0, 1)

    class Engines(dict):
        pass

    class Key(tuple):
        def __eq__(self, other):
            same = tuple.__eq__(self, other)
            engines["another"] = "engine of another problem"
            return same
        __hash__ = tuple.__hash__

    p, engines = problem, Engines()
    monkeypatch.setattr(evaluate, "_engines", engines)
    st = _structure_of(rpeg)
    key = Key((((st.name, st.memory_trainable),), tuple(sorted((m.value, s) for m, s in p.suite.specs.items())), p.workload, p.hw,
               p.device_space, p.K_eval, p.memory_policy, evaluate.RPEG_TRANSFER_RESOURCE_POLICY))
    engines[key] = "its engine"
    assert evaluate._engine_for(rpeg, p.suite, p.workload, p.hw, p.device_space, p.K_eval, p.memory_policy)[0] == "its engine"


def two_problems(monkeypatch):
    """Look-ups of the engines of two problems, of a table that calls `meanwhile` (in another thread, and goes on when that is
    done or waits) the first time `where` is reached."""
    (problem, [(rpeg, plan)]), (other, [(other_rpeg, _)]) = seeded(5, 0, 1), seeded(2, 0, 1)

    class Engine:
        def __init__(self, problem):
            self.problem = problem

    class Reversed:
        def __init__(self, engines):
            self.engines = engines

        def __reversed__(self):
            it = reversed(dict.items(self.engines))
            self.engines.reach("reversed")
            return it

    class Engines(dict):
        where, meanwhile, thread = None, None, None

        def reach(self, where):
            if where == self.where:
                self.where, self.taken = None, threading.Event()
                self.thread = threading.Thread(target=self.meanwhile)
                self.thread.start()
                self.taken.wait(0.3) if where == "found" else self.thread.join(0.3)

        def items(self):
            return Reversed(self)

        def pop(self, key):
            self.reach("found")
            got = dict.pop(self, key)
            if threading.current_thread() is self.thread:    # (the first thread goes on while the entry is out)
                self.taken.set()
                time.sleep(0.3)
            return got

    import rpeg_amd.engine.runtime as runtime
    engines = Engines()
    monkeypatch.setattr(runtime, "Engine", Engine)
    monkeypatch.setattr(evaluate, "_engines", engines)

    def look_up(p, r):
        return evaluate._engine_for(r, p.suite, p.workload, p.hw, p.device_space, p.K_eval, p.memory_policy)[0]
    return engines, lambda: look_up(problem, rpeg), lambda: look_up(other, other_rpeg)


def test_an_engine_is_looked_up_while_another_thread_changes_the_table(monkeypatch):
    engines, one, other = two_problems(monkeypatch)
    got = [one()]
    engines.where, engines.meanwhile = "reversed", lambda: got.append(other())
    assert one() is got[0]
    engines.thread.join()
    assert got[1] is other() and got[1] is not got[0]


def test_an_engine_that_another_thread_looks_up_too_is_the_same(monkeypatch):
    engines, one, other = two_problems(monkeypatch)
    want = one()
    other()
    got = []
    engines.where, engines.meanwhile = "found", lambda: got.append(one())
    assert one() is want
    engines.thread.join()
    assert got == [want]


def test_two_threads_that_make_an_engine_of_one_problem_get_the_same(monkeypatch):
    import rpeg_amd.engine.runtime as runtime
    _, one, _ = two_problems(monkeypatch)
    both, made = threading.Barrier(2), runtime.Engine

    def slow(problem):
        both.wait(10)
        return made(problem)
    monkeypatch.setattr(runtime, "Engine", slow)
    got = []
    threads = [threading.Thread(target=lambda: got.append(one())) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 2 and got[0] is got[1]
