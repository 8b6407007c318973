"""Positions of small tie-break classes of one size that follow one another, in the kernel that schedules a plan with two or four
lanes: counted together, a node's class found from its place in the run.  The oracle is the host build, bit for bit."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_positions import FREE_LINKS, same_bits


def test_a_place_in_a_run_tells_its_class():
    """... in floats, also where the reciprocal of the size is an ulp off."""
    place = np.arange(512, dtype=np.int32)
    for size in range(1, 65):
        exact = np.float32(1) / np.float32(size)
        for per_size in (np.nextafter(exact, np.float32(0)), exact, np.nextafter(exact, np.float32(2))):
            got = ((place.astype(np.float32) + np.float32(0.5)) * per_size).astype(np.int32)
            assert np.array_equal(got, place // size), (size, per_size)


@pytest.mark.gpu
@pytest.mark.parametrize("free", [False, True])
@pytest.mark.parametrize("c,K,n", [(2, 1, 9000), (2, 3, 33000), (2, 9, 17000), (5, 2, 33000), (5, 7, 9000), (4, 24, 9000), (3, 3, 9000)])
def test_runs_of_classes(c, K, n, free):
    """Runs of one class to two dozen, shorter than the lanes of a plan and longer than two turns of them; ranks that are all
    different and that are not."""
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, n)
    p = replace(cfg.problem, K_eval=K)
    if free:
        p = replace(p, hw=replace(p.hw, **FREE_LINKS))
    want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16)
    eng = Engine(p)
    eng.set_state_lanes(4)
    try:
        for call in range(3):
            out = eng.eval(batch, gate_stale=True)
            assert eng.stats()["quad_tasks"] > 0
            assert np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want[k]), (k, call)
    finally:
        eng.close()
