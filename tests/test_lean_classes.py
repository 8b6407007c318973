"""Classes lowered for the calls of a wavefront per plan, without what only the kernel of a few lanes per plan keeps of them
(rpeg_lower.h: Lowering::run), and lowered once more when a batch for that kernel meets them."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_class_blob import HDR, check_blob
from tests.test_shared_rows import same_bits


@pytest.mark.parametrize("c,K", [(1, 4), (1, 12), (2, 4), (3, 6), (4, 1), (5, 4)])
def test_a_lean_class_is_the_full_one_without_its_last_sections(c, K):
    cfg, batch = seeded_batch(c, 400)
    port = CpuPort(replace(cfg.problem, K_eval=K))
    sigs = np.unique(port.eval(batch)["sig"])
    for sig in sigs[sigs != np.uint64(2 ** 64 - 1)][:40]:
        full, edges = port.blob(sig)
        lean, edges2 = port.blob(sig, few_lanes=False)
        assert np.array_equal(lean, port.blob(sig, few_lanes=False, own=True)[0]) and np.array_equal(edges, edges2)
        check_blob(lean, edges)
        n_words = len(HDR) + 4
        wf, wl = full[:4 * n_words].view("<u4").tolist(), lean[:4 * n_words].view("<u4").tolist()
        n_rows, n_types, off_qrec, off_type = wl[len(HDR):]
        assert (n_rows, n_types) == (0, 0) and off_qrec == off_type == wf[len(HDR) + 2]
        assert len(lean) == (off_qrec + 15) // 16 * 16 and len(full) >= len(lean) + 4 * wf[0] - 16
        b = HDR.index("bytes")
        assert [x for k, x in enumerate(wl[:len(HDR)]) if k != b] == [x for k, x in enumerate(wf[:len(HDR)]) if k != b]
        assert np.array_equal(lean[4 * n_words:off_qrec], full[4 * n_words:off_qrec])


@pytest.mark.gpu
@pytest.mark.parametrize("c,K,few,many,lanes", [(5, 4, 900, 20011, -1), (4, 1, 200, 16384, -1), (2, 4, 9000, 17000, -1), (3, 6, 300, 3000, 4)])
def test_a_batch_for_a_few_lanes_per_plan_behind_calls_that_lowered_its_classes_lean(c, K, few, many, lanes):
    from rpeg_amd.engine.runtime import Engine
    cfg, small = seeded_batch(c, few)
    _, large = seeded_batch(c, many)
    p = replace(cfg.problem, K_eval=K)
    port = CpuPort(p)
    want_small = port.eval(small, flags=abi.GATE_STALE, threads=16)
    want_large = port.eval(large, flags=abi.GATE_STALE, threads=16)
    eng = Engine(p)
    try:
        for turn in range(2):
            eng.set_state_lanes(-1)
            out = eng.eval(small, gate_stale=True)
            assert np.array_equal(out["mask"], want_small["mask"])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want_small[k]), (turn, k)
            eng.set_state_lanes(lanes)
            took = 0
            for call in range(4):   # (the first ones measure the classes)
                out = eng.eval(large, gate_stale=True)
                took += eng.stats()["quad_tasks"]
                assert np.array_equal(out["mask"], want_large["mask"])
                for k in ("makespan", "peak", "score"):
                    assert same_bits(out[k], want_large[k]), (turn, call, k)
            assert took > 0
    finally:
        eng.close()
