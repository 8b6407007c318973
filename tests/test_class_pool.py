"""The class pool on the device: blobs go there in stretches (one class after the other in small calls, a stretch per
lowering thread in large ones), and a pool that outgrows its allocation moves.  Classes of every stretch, from before and
after a move, give the host build's bits; and what a call lowered is counted by the call that did it."""

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd import configs
from rpeg_amd.engine import abi
from rpeg_amd.search import candidates
from tests.helpers import seeded_batch

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


def test_classes_of_every_stretch_survive_the_pool_s_moves():
    from rpeg_amd.engine.runtime import Engine
    cfg = configs.config(3)                      # (some 7 KB a class: the first megabyte holds 150 of them)
    p = cfg.problem
    port, eng = CpuPort(p), Engine(p)
    try:
        seen = []
        # small batches (class after class), large ones (threads), small again: each adds classes, all are asked again
        for k, n in enumerate((3, 60, 2, 1500, 40, 9000, 1, 30)):
            batch = candidates.generate(p, n, cfg.tau_choices, seed=900 + k, tag=3)
            seen.append((batch, port.eval(batch, flags=abi.GATE_STALE, threads=16)))
            for b, ref in seen:
                out = eng.eval(b, gate_stale=True)
                assert np.array_equal(out["mask"], ref["mask"]), (k, b.n)
                for f in ("makespan", "peak", "score"):
                    assert same_bits(out[f], ref[f]), (k, b.n, f)
        eng.reset_classes()
        for b, ref in seen[::-1]:
            assert same_bits(eng.eval(b, gate_stale=True)["score"], ref["score"])
    finally:
        eng.close()


def test_a_call_counts_the_classes_it_lowers():
    """rpeg_engine_stats: also where one plan is evaluated with its trace, which lowers a class not met before once."""
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(1, 12)
    eng, port = Engine(cfg.problem), CpuPort(cfg.problem)
    try:
        sig, known = port.eval(batch)["sig"], set()
        for i in range(batch.n):
            if sig[i] == np.uint64(2 ** 64 - 1):
                continue
            eng.trace(batch, i)
            assert eng.stats()["classes_lowered"] == (0 if sig[i] in known else 1), i
            known.add(sig[i])
            eng.trace(batch, i)
            assert eng.stats()["classes_lowered"] == 0
        out = eng.eval(batch, gate_stale=True)
        assert eng.stats()["classes_lowered"] == 0
        assert same_bits(out["score"], port.eval(batch, flags=abi.GATE_STALE)["score"])
    finally:
        eng.close()
