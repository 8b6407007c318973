"""Batches of more plans per compute unit than k_quad's forms find room for at once, of large graphs: launches by LDS, ready sets
of up to 24 entries a plan.  The oracle is the host build, bit for bit."""

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_positions import same_bits

pytestmark = pytest.mark.gpu

DEEP_PLANS = 512   # a compute unit: more of them make a batch deep


@pytest.mark.parametrize("per_cu,more,deep", [(DEEP_PLANS, 1, True), (586, 0, True), (DEEP_PLANS, 0, False)])
def test_large_graphs_in_a_deep_batch(per_cu, more, deep):
    import torch
    from rpeg_amd.engine.runtime import Engine
    n = torch.cuda.get_device_properties(0).multi_processor_count * per_cu + more
    cfg, batch = seeded_batch(3, n)
    want = CpuPort(cfg.problem).eval(batch, flags=abi.GATE_STALE, threads=16, want_mass=True)
    eng = Engine(cfg.problem)

    def launches():
        st = eng.stats()
        return [st[f"quad_launches_{k}"] for k in (8, 16, 24)]

    try:
        for call in range(5):   # (by what the main kernel has measured from the second or third on)
            out = eng.eval(batch, gate_stale=True)
            assert np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want[k]), (k, call)
        assert eng.stats()["quad_plans"] > n // 2
        if deep:   # measured classes in the form of 24 entries, which others leave to k_plan, and launches by LDS
            assert launches()[2] > 1 and max(launches()[:2]) > 2, launches()
        else:
            assert launches()[2] <= 1 and max(launches()[:2]) <= 2, launches()
        # with masses (more LDS per plan: other bins); the main kernel would take such a batch, so a margin that leaves it none
        eng.set_split_model([9.0, 0.8, 10.0, 1.3, 0.2, 0.65, 0.01, 0.97, 0.98, 1.25])
        mass = eng.eval(batch, gate_stale=True, mass=True)
        assert np.array_equal(mass["mask"], want["mask"])
        for k in ("makespan", "peak", "score", "mass"):
            assert same_bits(mass[k], want[k]), k
        assert eng.stats()["quad_plans"] > n // 2
        if deep:
            assert launches()[2] > 1 and max(launches()[:2]) > 2, launches()
    finally:
        eng.close()
