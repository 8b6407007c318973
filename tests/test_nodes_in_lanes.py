"""The scheduler that gives every node a lane, or a half or third of one, at the sizes where its form changes: 64, 128 and
192 lowered nodes and their neighbours.  The oracle is the host build, which schedules with an ordered list; makespan, peak,
score, mask and critical-chain mass are its bits, the utilisation that of the single-plan trace."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch

pytestmark = pytest.mark.gpu

# workload, unrolled steps, node counts that the 400 plans have among others
EDGES = [(1, 5, {63, 64, 127, 128}), (1, 3, {64, 66}), (3, 6, {64, 128, 129, 130}), (3, 7, {129, 192, 194}), (1, 12, {191})]


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


@pytest.mark.parametrize("c,K,edges", EDGES)
def test_graphs_at_the_edges_of_a_form(c, K, edges):
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, 400)
    p = replace(cfg.problem, K_eval=K)
    port = CpuPort(p)
    want = port.eval(batch, flags=abi.GATE_STALE, threads=16, want_mass=True)
    nodes = {i: len(port.lower(batch, i)["kind"]) for i in range(batch.n) if want["mask"][i]}
    assert edges <= set(nodes.values())
    eng = Engine(p)
    eng.set_state_lanes(1)
    try:
        for _ in range(3):   # (the lane masks are built anew by every launch)
            for out in (eng.eval(batch, gate_stale=True), eng.eval_mass(batch, gate_stale=True), eng.eval_util(batch, gate_stale=True)):
                assert np.array_equal(out["mask"], want["mask"])
                assert all(same_bits(out[k], want[k]) for k in ("makespan", "peak", "score"))
                assert "mass" not in out or same_bits(out["mass"], want["mass"])
        for n in edges:
            i = next(i for i, m in nodes.items() if m == n)
            assert float(out["util"][i]).hex() == float(eng.trace_metrics(batch, i)[0]).hex(), n
    finally:
        eng.close()
