"""Ready sets that outgrow their form of the few-lanes-per-plan kernel: the class's statistic says so, and its plans have
room in the calls that follow.  (Forms of 8, 16 and 24 entries, by the longest ready set that the class's earlier plans
had; a plan with more is redone by the launch that ends the call.)"""

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


@pytest.mark.parametrize("c,n,lanes", [(5, 20011, -1), (5, 20011, 4), (1, 17001, 4)])
def test_plans_that_outgrow_their_form_have_room_in_the_next_calls(c, n, lanes):
    """Forms learned from one batch, then another batch of the same classes whose plans have longer ready sets: its first
    call redoes some of them, and no call redoes any once a class has gone through the forms (two steps at most, one per
    call).  stats()["redone_before"] speaks of the call before."""
    from rpeg_amd.engine.runtime import Engine
    cfg, a = seeded_batch(c, n)
    _, b = seeded_batch(c, n, start=n)
    ref = CpuPort(cfg.problem).eval(b, flags=abi.GATE_STALE, threads=16)
    eng = Engine(cfg.problem)
    eng.set_state_lanes(lanes)
    try:
        for _ in range(6):
            eng.eval(a, gate_stale=True)
        redone = []
        for call in range(7):
            out = eng.eval(b, gate_stale=True)
            redone.append(eng.stats()["redone_before"])
            assert eng.stats()["quad_tasks"] > 0
            assert np.array_equal(out["mask"], ref["mask"]), call
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], ref[k]), (call, k)
        assert max(redone[1:]) > 0, redone        # (the batches do what the test is about)
        assert redone[4:] == [0, 0, 0], redone    # the calls from the fourth on
    finally:
        eng.close()


def test_a_small_batch_between_takes_over_what_the_plans_needed():
    """The same with batches of a wavefront per plan between the large ones: they are the calls that hear of the redone plans
    (and that leave nothing of it for the next), so they hand over the classes' ready sets too."""
    from rpeg_amd.engine.runtime import Engine
    cfg, a = seeded_batch(5, 20011)
    _, b = seeded_batch(5, 20011, start=20011)
    ref = CpuPort(cfg.problem).eval(b, flags=abi.GATE_STALE, threads=16)
    eng = Engine(cfg.problem)
    try:
        eng.set_state_lanes(1)      # (every class is lowered, no ready set measured)
        eng.eval(b, gate_stale=True)
        eng.eval(a, gate_stale=True)
        eng.set_state_lanes(-1)
        for _ in range(6):
            eng.eval(a, gate_stale=True)
        redone = []
        for call in range(6):
            out = eng.eval(b, gate_stale=True)
            assert eng.stats()["quad_tasks"] > 0
            assert np.array_equal(out["mask"], ref["mask"]), call
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], ref[k]), (call, k)
            eng.eval(a.slice(0, 6000), gate_stale=True)
            assert eng.stats()["state_lanes"] == 1 and eng.stats()["classes_lowered"] == 0
            redone.append(eng.stats()["redone_before"])
        assert redone[0] > 0, redone              # (the batches do what the test is about)
        assert redone[3:] == [0, 0, 0], redone
    finally:
        eng.close()
