"""The settings of the split between the scheduling kernels: what they bound, and that no bit depends on them."""

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


@pytest.mark.parametrize("c,n", [(2, 65536), (5, 20011), (4, 16384)])
def test_the_share_bounds_what_the_few_lanes_kernel_takes(c, n):
    """rpeg_engine_set_quad_share: at most that many percent of the plans (4, 16384: a batch too small for the main
    kernel's full wavefronts, which moves whole or not at all); the rest runs in the main kernel beside it."""
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, n)
    ref = CpuPort(cfg.problem).eval(batch, flags=abi.GATE_STALE, threads=16, want_mass=True)
    eng, took = Engine(cfg.problem), {}
    try:
        for share in (100, 10, 40, 100, 0):
            eng.set_quad_share(share)
            for call in range(4):
                out = eng.eval(batch, gate_stale=True, mass=(call == 3))
                st = eng.stats()
                assert st["quad_plans"] * 100 <= n * share, (share, call, st)
                assert np.array_equal(out["mask"], ref["mask"]), (share, call)
                for k in ("makespan", "peak", "score") + (("mass",) if call == 3 else ()):
                    assert same_bits(out[k], ref[k]), (share, call, k)
            took[share] = st["quad_plans"]
    finally:
        eng.close()
    if n > 16384:
        assert 0 < took[10] < took[40] < took[100], took
    else:
        assert took[10] == took[40] == 0 < took[100], took


def test_all_ten_figures_can_be_set():
    """rpeg_engine_set_split_model: the tenth, what a graph of more than 128 nodes costs k_plan, made dear and free: what
    moves is where plans run.  AC-share plans, most of them of more than 128 nodes, k_plan made to look cheap."""
    from rpeg_amd.engine.runtime import Engine, EngineError
    cfg, batch = seeded_batch(3, 17003)
    ref = CpuPort(cfg.problem).eval(batch, flags=abi.GATE_STALE, threads=16)
    eng, solo = Engine(cfg.problem), []
    try:
        for tenth in (0.1, 50.0):
            eng.set_split_model([12.0, 0.9, 10.0, 1.3, 0.2, 0.65, 1.15, 0.97, 0.98, tenth])
            for _ in range(4):
                out = eng.eval(batch, gate_stale=True)
                assert np.array_equal(out["mask"], ref["mask"]) and same_bits(out["score"], ref["score"])
            solo.append(eng.stats()["single_plan_tasks"])
        assert solo[0] > solo[1], solo
        for wrong in (8, 11):
            with pytest.raises(EngineError):
                eng.set_split_model([1.0] * wrong)
    finally:
        eng.close()
