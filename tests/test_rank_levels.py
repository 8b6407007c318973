"""The rank pass and the critical chain of the kernel that gives a plan one or four wavefronts, where their forms change: graphs of
more levels than a wavefront has lanes, of more nodes than it has, chains of up to six quantiles, and graphs too small for the
walk in stretches; scores and masses of the host build bit for bit (a rank decides ties, a
mass is summed in the order of the walk)."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from tests.helpers import seeded_batch
from tests.test_class_blob import HDR
from tests.test_class_pool import same_bits

CASES = [(1, 1), (1, 4), (1, 14), (2, 1), (2, 4), (2, 16), (3, 5), (4, 1), (4, 4), (4, 33), (5, 4), (5, 9)]


def headers(c, K, n):
    cfg, batch = seeded_batch(c, n)
    port = CpuPort(replace(cfg.problem, K_eval=K))
    sigs = np.unique(port.eval(batch)["sig"])
    for sig in sigs[sigs != np.uint64(2 ** 64 - 1)]:
        blob, _ = port.blob(sig)
        yield dict(zip(HDR, blob[:4 * len(HDR)].view("<u4").tolist()))


def test_the_cases_have_what_they_are_for():
    levels, nodes = set(), set()
    for c, K in CASES:
        for h in headers(c, K, 60):
            if h["n_nodes"] > 384:
                continue
            nodes.add(h["n_nodes"])
            levels.add(h["n_levels"])
    assert min(nodes) <= 32 < max(nodes) and any(n > 192 for n in nodes)
    assert min(levels) < 62 < max(levels)


@pytest.mark.gpu
@pytest.mark.parametrize("c,K", CASES)
@pytest.mark.parametrize("n", [60, 2500])   # four wavefronts a plan, and one
def test_scores_and_masses(c, K, n):
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, n)
    p = replace(cfg.problem, K_eval=K)
    want = CpuPort(p).eval(batch, threads=16, want_mass=True)
    eng = Engine(p)
    try:
        out = eng.eval_mass(batch)
        assert np.array_equal(out["mask"], want["mask"])
        for k in ("makespan", "peak", "score", "mass"):
            assert same_bits(out[k], want[k]), k
    finally:
        eng.close()
