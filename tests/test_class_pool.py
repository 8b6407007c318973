"""What a call lowered is counted by the call that did it."""

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch

pytestmark = pytest.mark.gpu


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


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
