"""Ready-time rows shared by nodes that never need one at the same time, reservations by type, and the word per node that
names them (rpeg_class.h: QuadRec): derived again from the edge list, and the kernel that keeps only these per plan, with the
ranks of all of a wavefront's plans at once (few wavefronts) and of a quarter at a time (many), against the host build."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_class_blob import HDR, NODE


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


@pytest.mark.parametrize("c,K", [(1, 4), (1, 12), (2, 4), (3, 4), (4, 1), (5, 4)])
def test_nodes_of_a_row_come_one_after_the_other(c, K):
    cfg, batch = seeded_batch(c, 400)
    port = CpuPort(replace(cfg.problem, K_eval=K))
    sigs = np.unique(port.eval(batch)["sig"])
    for sig in sigs[sigs != np.uint64(2 ** 64 - 1)][:40]:
        blob, edges = port.blob(sig)
        words = blob[:4 * (len(HDR) + 4)].view("<u4").tolist()
        h = dict(zip(HDR, words))
        n_rows, n_types, off_qrec, off_type = words[len(HDR):]
        n = h["n_nodes"]
        node = blob[h["off_node"]:h["off_node"] + 8 * n].view(NODE)
        place = blob[h["off_place"]:h["off_place"] + 2 * n].view("<u2")
        topo = blob[h["off_topo"]:h["off_topo"] + 2 * n].view("<u2").tolist()
        q = blob[off_qrec:off_qrec + 4 * n].view("<u4")[place].astype(np.int64)   # by node
        types = blob[off_type:off_type + 2 * n_types].view("<u2")
        assert off_type + 2 * n_types <= h["bytes"] and 1 <= n_rows <= 128 and 1 <= n_types <= 64
        assert np.array_equal(q & 7, np.minimum(node["n_succ"], 7)) and np.array_equal((q >> 3) & 63, node["indeg"])
        assert np.array_equal((q >> 10) & 255, node["slot"])
        assert np.array_equal(types[(q >> 18) & 63], node["blocked"].astype(int) | node["cond"].astype(int) << 8)
        row = (q >> 24) & 127
        assert row.max() < n_rows and np.array_equal(row == 0, node["indeg"] < 2)
        pred = [[] for _ in range(n)]
        for a, b in edges:
            pred[b].append(int(a))
        anc = [set() for _ in range(n)]
        for v in topo:
            for a in pred[v]:
                anc[v] |= anc[a] | {a}
        last = {}
        for y in topo:
            if row[y]:
                x = last.get(row[y])
                assert x is None or all(set(pred[x]) <= anc[p] for p in pred[y])
                last[row[y]] = y


@pytest.mark.gpu
@pytest.mark.parametrize("c,K,n", [(4, 1, 33), (1, 12, 500), (3, 6, 200), (3, 6, 5000), (5, 4, 20000)])
def test_ranks_of_all_and_of_a_quarter_of_the_plans(c, K, n):
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, n)
    p = replace(cfg.problem, K_eval=K)
    want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16, want_mass=True)
    eng = Engine(p)
    eng.set_state_lanes(4)
    try:
        for call in range(5):   # (24 entries first, then by what the plans had)
            out = eng.eval(batch, gate_stale=True, mass=call == 4)
            assert eng.stats()["quad_tasks"] > 0 and np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score") + (("mass",) if call == 4 else ()):
                assert same_bits(out[k], want[k]), (call, k)
    finally:
        eng.close()
