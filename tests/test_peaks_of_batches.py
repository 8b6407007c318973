"""The memory-model launch of large batches (three, four and six vertices to a structure, plans whose vertices first appear in
another order than their own among them, a last block that is not full): largest device peaks, gate bits and penalties of the
host build bit for bit, under both memory models and with a limit on worker groups."""

import dataclasses

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from rpeg_amd.model.memory import MemoryPolicy
from tests.helpers import seeded_batch
from tests.test_class_pool import same_bits
from tests.test_coresident_golden import coresident_problem
from tests.test_one_wavefront_batches import broken


@pytest.mark.gpu
@pytest.mark.parametrize("policy", [{}, dict(max_worker_groups_per_gpu=3, worker_overhead_bytes=1 << 30), dict(optimizer_stage=1)])
@pytest.mark.parametrize("coresident", [False, True])
@pytest.mark.parametrize("c,n", [(1, 13825), (2, 13824), (3, 13823), (4, 14001)])
def test_peaks_beside_the_scheduling_kernels(c, n, coresident, policy):
    from rpeg_amd.engine.runtime import DeviceBatch, Engine
    cfg, batch = seeded_batch(c, n)
    p = cfg.problem
    p = coresident_problem(p, policy, p.K_eval) if coresident else dataclasses.replace(p, memory_policy=MemoryPolicy(**policy))
    assert (batch.head[1] > 0).any() or c == 4            # phases: what lets a vertex appear out of turn
    broken(batch, 41)
    want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16)
    assert len(np.unique(want["peak"][np.isfinite(want["peak"])])) > 50
    eng = Engine(p)
    try:
        out = eng.eval_device(DeviceBatch(batch, "cuda:0"))
        assert eng.stats()["state_lanes"] != 1
        assert np.array_equal(out["mask"].cpu().numpy(), want["mask"])
        for k in ("peak", "score", "makespan"):
            assert same_bits(out[k].cpu().numpy(), want[k]), k
    finally:
        eng.close()
