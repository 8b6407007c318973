"""What the kernel of a few lanes per plan reads in its rank pass (rpeg_class.h: RankRec): levels computed one after the other in the
rows that nodes share give the ranks that the edge list gives; and that kernel where all plans' ranks lie in LDS and where they
go through memory by parts, with the host build's bits (the ranks decide the order of every tie)."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_class_blob import HDR, NODE, ORDER
from tests.test_class_pool import same_bits

RANK = np.dtype([("succ", "u1", 4), ("row", "u1"), ("slot", "u1"), ("id", "<u2")])


@pytest.mark.parametrize("c,K", [(1, 4), (1, 12), (2, 4), (3, 4), (3, 7), (4, 1), (4, 16), (5, 4)])
def test_ranks_in_shared_rows_are_the_longest_paths(c, K):
    cfg, batch = seeded_batch(c, 400)
    port = CpuPort(replace(cfg.problem, K_eval=K))
    sigs = np.unique(port.eval(batch)["sig"])
    rng = np.random.default_rng(7)
    taken = 0
    for sig in sigs[sigs != np.uint64(2 ** 64 - 1)][:40]:
        blob, edges = port.blob(sig)
        words = blob[:4 * (len(HDR) + 4)].view("<u4").tolist()
        h = dict(zip(HDR, words))
        n_rows, off_qrec = words[len(HDR)], words[len(HDR) + 2]
        if n_rows == 0:
            continue
        taken += 1
        n = h["n_nodes"]
        at = off_qrec + (4 * n + 7) // 8 * 8
        rec = blob[at:at + 8 * (n + 2)].view(RANK)
        used = int(rec["id"][n + 1])
        assert 2 <= used <= 256 and rec["id"][n] == n and rec["row"][n] == 1 and not rec["succ"][n].any()
        node = blob[h["off_node"]:h["off_node"] + 8 * n].view(NODE)
        place = blob[h["off_place"]:h["off_place"] + 2 * n].view("<u2").astype(int)
        orec = blob[h["off_orec"]:h["off_orec"] + 8 * n].view(ORDER)
        lbeg = blob[h["off_lbeg"]:h["off_lbeg"] + 2 * (h["n_levels"] + 1)].view("<u2").tolist()
        id_of = np.empty(n, int)
        id_of[orec["at"]] = np.arange(n)            # by place
        succ = [[] for _ in range(n)]
        for a, b in edges:
            succ[a].append(int(b))
        by_place = np.empty(n, int)
        by_place[place] = np.arange(n)
        dur = rng.random(n)                         # per node
        want = np.zeros(n)
        for v in by_place:
            want[v] = dur[v] + max([want[w] for w in succ[v]], default=0.0)
        rows = np.full(used, np.nan)
        rows[0] = 0.0
        got = np.zeros(n)
        for lo, hi in zip(lbeg, lbeg[1:]):
            # (a level's lanes may take any of its nodes first: what one writes no other of the level reads)
            for k in rng.permutation(np.arange(lo, hi)):
                r, v = rec[k], by_place[k]
                assert r["slot"] == node["slot"][v] and (int(r["id"]) & 0x1FF) == id_of[k]
                assert bool(int(r["id"]) & 0x8000) == (len(succ[v]) > 4)
                read = [int(x) for x in r["succ"]] + [int(rec[place[w]]["row"]) for w in succ[v][4:]]
                got[v] = dur[v] + max(rows[read])
                assert 0 < r["row"] < used
                if r["row"] > 1:
                    rows[r["row"]] = got[v]
        assert np.array_equal(got, want)
    assert taken


@pytest.mark.gpu
@pytest.mark.parametrize("c,K,n", [(4, 4, 33), (4, 4, 70001), (4, 16, 3001), (2, 4, 1000), (2, 4, 40001), (5, 4, 777), (5, 4, 30011), (3, 6, 15001)])
def test_ranks_at_once_and_by_parts(c, K, n):
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, n)
    p = replace(cfg.problem, K_eval=K)
    want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16)
    eng = Engine(p)
    try:
        eng.set_state_lanes(4)
        for call in range(3):   # (24 entries first, then by what the plans had)
            out = eng.eval(batch, gate_stale=True)
            assert eng.stats()["quad_tasks"] > 0 and np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want[k]), (call, k)
    finally:
        eng.close()


@pytest.mark.gpu
@pytest.mark.parametrize("c,n,nbytes", [(4, 140001, 1), (2, 70001, 1 << 20), (5, 60011, 3 << 20)])
def test_ranks_by_turns(c, n, nbytes):
    """Less memory for ranks than the launches' tasks take at once (1 byte: one task of each launch at a time)."""
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, n)
    want = CpuPort(cfg.problem).eval(batch, flags=abi.GATE_STALE, threads=16)
    eng = Engine(cfg.problem)
    try:
        eng.set_state_lanes(4)
        for most in (0, nbytes, 0):
            eng.set_rank_memory(most)
            out = eng.eval(batch, gate_stale=True)
            assert eng.stats()["quad_tasks"] > 0 and np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score"):
                assert same_bits(out[k], want[k]), (most, k)
    finally:
        eng.close()


@pytest.mark.gpu
def test_a_batch_with_slightly_larger_graphs_needs_no_new_memory():
    import torch
    from rpeg_amd.engine.runtime import DeviceBatch, Engine
    cfg, batch = seeded_batch(5, 60011)
    port = CpuPort(cfg.problem)
    sig = port.eval(batch, threads=16)["sig"]
    known, of = np.unique(sig[sig != np.uint64(2 ** 64 - 1)], return_inverse=True)
    nodes = np.array([port.blob(x)[0][:4].view("<u4")[0] for x in known])[of]
    by_size = np.flatnonzero(sig != np.uint64(2 ** 64 - 1))[np.argsort(nodes, kind="stable")]
    n = 40000
    # mostly plans of the smallest graphs, with some of the next larger (up to 132 nodes), and with fewer of the largest (158)
    first, second = (np.concatenate([by_size[:n - n // k], by_size[at:at + n // k]]) for at, k in ((44000, 3), (56000, 10)))
    eng = Engine(cfg.problem)
    try:
        eng.set_state_lanes(4)
        out = eng.alloc_outputs(n)
        for _ in range(3):                          # every class is lowered and has its form
            for k in range(6):
                eng.eval_device(DeviceBatch(batch.take(by_size[k::6]), "cuda:0"), out)
        batches = [DeviceBatch(batch.take(idx), "cuda:0") for idx in (first, second)]
        free = []
        for b in batches:
            for _ in range(2):
                eng.eval_device(b, out)
            torch.cuda.synchronize()
            free.append(torch.cuda.mem_get_info()[0])
        assert free[0] == free[1]
        eng.set_rank_memory(8)                      # (gives back what it holds: there was some)
        assert torch.cuda.mem_get_info()[0] > free[1]
    finally:
        eng.close()
