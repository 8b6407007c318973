"""Latencies below zero (Hardware.alpha_*: an intercept fitted to measurements may be) make transfers of small payloads end before
they start, and operators too.  The kernel of a few lanes per plan shares ready-time rows, which it then sets back when they
have been read, and gives a chain's nodes the largest rank instead of the first one's.  Held to the
host build, without a plan redone for it.  (Not to the reference, whose devices become available again when the last node on them
ends, earlier than another where that node ends before it starts: here availability only grows, on every path.)"""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_shared_rows import same_bits


def problem(c, K, alpha):
    p = seeded_batch(c, 1)[0].problem
    return replace(p, K_eval=K, hw=replace(p.hw, alpha_p2p_g=alpha, alpha_p2p_n=alpha, alpha_p2p_r=alpha))


@pytest.mark.parametrize("c,K,alpha", [(1, 4, -0.02), (3, 6, -0.02), (4, 1, -5.0), (5, 4, -5.0)])
def test_such_plans_exist(c, K, alpha):
    p = problem(c, K, alpha)
    _, batch = seeded_batch(c, 24)
    port = CpuPort(p)
    out = port.eval(batch)
    low = [port.lower(batch, i) for i in range(24)]
    assert sum(bool((x["dur"] < 0.0).any()) for x in low) > 4 and (out["mask"] & abi.MASK_ERROR == 0).all()
    assert not same_bits(out["makespan"], CpuPort(replace(p, hw=seeded_batch(c, 1)[0].problem.hw)).eval(batch)["makespan"])


@pytest.mark.parametrize("c,K,alpha,least", [(1, 4, -0.02, 30), (3, 6, -0.02, 25), (5, 4, -5.0, 40)])
def test_chains_that_shrink_exist(c, K, alpha, least):
    _, batch = seeded_batch(c, 64)
    port = CpuPort(problem(c, K, alpha))
    low = [port.lower(batch, i) for i in range(64)]
    assert sum(bool(((x["kind"] == 0) & (x["step"] < K - 1) & (x["dur"] < 0.0)).any()) for x in low) >= least


@pytest.mark.gpu
@pytest.mark.parametrize("c,K,n,lanes", [(1, 4, 500, 4), (1, 4, 500, 1), (3, 6, 700, 4), (4, 1, 33, 4), (4, 1, 16384, -1), (5, 4, 20000, -1)])
@pytest.mark.parametrize("alpha", [-0.02, -5.0])
def test_plans_that_shrink_in_the_kernel_of_a_few_lanes(c, K, n, lanes, alpha):
    from rpeg_amd.engine.runtime import Engine
    p = problem(c, K, alpha)
    _, batch = seeded_batch(c, n)
    want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16, want_mass=True)
    eng = Engine(p)
    eng.set_state_lanes(lanes)
    took = redone = 0
    try:
        for call in range(4):
            out = eng.eval(batch, gate_stale=True, mass=call == 3)
            took += eng.stats()["quad_plans"]
            redone += eng.stats()["redone_before"]
            assert np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score") + (("mass",) if call == 3 else ()):
                assert same_bits(out[k], want[k]), (call, k)
        assert (took > 0) == (lanes != 1)
        assert redone * 50 <= took   # (ready sets that outgrew their lanes, if any)
    finally:
        eng.close()
