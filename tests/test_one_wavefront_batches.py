"""Batches of a wavefront per plan (more than four and at most 52 plans per compute unit, with the edges of that range and of the
blocks of 64 and 256 plans), in the plans' own order up to eight per compute unit and for few classes, else dealt to their tasks on the
device, with durations ahead of those of more than sixteen and of those dealt, and of four wavefronts: outputs and masks of the host build bit for bit, plans that break a rule and
plans of both structures among them, critical-chain masses too, on an engine that has met none, some and all of the classes."""

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_class_pool import same_bits


def broken(batch, every):
    """Every so-manieth plan breaks an integer rule."""
    batch.vert[2, ::every] = 3        # tp of the first vertex
    return batch


@pytest.mark.gpu
@pytest.mark.parametrize("c,n", [(1, 1), (2, 1023), (3, 1024), (1, 1025), (1, 2048), (1, 2049), (2, 4097), (2, 8191), (3, 3000), (4, 1100), (4, 13311), (5, 13312)])
def test_a_wavefront_per_plan(c, n):
    from rpeg_amd.engine.runtime import DeviceBatch, Engine
    cfg, first = seeded_batch(c, n)
    _, second = seeded_batch(c, n, start=n // 2)          # half of it new
    port = CpuPort(cfg.problem)
    eng = Engine(cfg.problem)
    try:
        for batch in (broken(first, 37), second, first):
            want = port.eval(batch, flags=abi.GATE_STALE, threads=16)
            assert n < 500 or (want["mask"] == 0).any() == (batch is first)
            out = eng.eval_device(DeviceBatch(batch, "cuda:0"))
            assert n == 1 or eng.stats()["state_lanes"] == 1
            assert np.array_equal(out["mask"].cpu().numpy(), want["mask"])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k].cpu().numpy(), want[k]), k
        masses = eng.eval_mass(first)
        small = {k: np.concatenate([eng.eval_mass(first.slice(i, min(i + 500, n)))[k] for i in range(0, n, 500)]) for k in ("mass", "score")}
        for k in small:
            assert same_bits(masses[k], small[k]), k
    finally:
        eng.close()
