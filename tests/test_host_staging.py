"""Host-pointer batches that are staged in chunks through pinned memory: sizes at the edges of a chunk (512 KiB, of fields and of
results) and of its sixteen-byte copies, several rounds of the four pinned chunks, odd ones, rows apart from each other by more than the batch, with and without masses,
larger and smaller calls in turn on one engine, calls that want some or none of the results between them; outputs of the host build
bit for bit."""

import ctypes as C

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_class_pool import same_bits


@pytest.mark.gpu
@pytest.mark.parametrize("c,sizes", [(4, (1025, 26214, 26215, 1031)), (2, (2049, 20971, 20973, 5243)), (1, (8738, 1027)), (4, (131071, 34953, 32768)), (3, (60001, 17478))])
def test_staged_batches(c, sizes):
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, max(sizes))
    port = CpuPort(cfg.problem)
    want = port.eval(batch, flags=abi.GATE_STALE, threads=16)
    eng = Engine(cfg.problem)
    try:
        for n in sizes:
            out = eng.eval(batch.slice(0, n))
            assert np.array_equal(out["mask"], want["mask"][:n])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want[k][:n]), (n, k)
        n, stride = min(sizes), max(sizes)          # rows of the whole batch, outputs wanted in part
        vert, head = np.ascontiguousarray(batch.vert), np.ascontiguousarray(batch.head)
        assert vert.shape[1] == stride
        soa = abi.PlanSoaT(vert.ctypes.data, head.ctypes.data, stride)
        score = np.full(n + 1, -1.0)
        assert eng.lib.rpeg_eval_host(eng._h, n, C.addressof(soa), abi.GATE_STALE, None, None, score.ctypes.data, None, None, None) == 0
        assert same_bits(score[:n], want["score"][:n]) and score[n] == -1.0
        masses = eng.eval_mass(batch.slice(0, n))["mass"]
        assert same_bits(masses, eng.eval_mass_device(batch.slice(0, n))["mass"])
    finally:
        eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n_between", [1500, 30001])      # results in one piece, and one by one
@pytest.mark.parametrize("wanted", [(), ("makespan",), ("mask",)])
def test_calls_that_want_few_results_or_none(n_between, wanted):
    """The pinned chunks are at rest when a call returns: the plans of the next one go there at once."""
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(2, 30001)
    want = CpuPort(cfg.problem).eval(batch, flags=abi.GATE_STALE, threads=16)
    vert, head = np.ascontiguousarray(batch.vert), np.ascontiguousarray(batch.head)
    eng = Engine(cfg.problem)
    try:
        for first in (0, 9001, 18002):
            few = {k: np.zeros(n_between, np.uint8 if k == "mask" else np.float64) for k in wanted}
            soa = abi.PlanSoaT(vert.ctypes.data, head.ctypes.data, vert.shape[1])
            ptr = [few[k].ctypes.data if k in few else None for k in ("makespan", "peak", "score", "mask")]
            assert eng.lib.rpeg_eval_host(eng._h, n_between, C.addressof(soa), abi.GATE_STALE, *ptr, None, None) == 0
            out = eng.eval(batch.slice(first, first + 9001))
            assert np.array_equal(out["mask"], want["mask"][first:first + 9001])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want[k][first:first + 9001]), k
            for k in few:
                assert np.array_equal(few[k], want[k][:n_between]) if k == "mask" else same_bits(few[k], want[k][:n_between]), k
    finally:
        eng.close()
