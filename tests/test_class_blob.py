"""The tables of a lowered class (rpeg_class.h: ClassHdr and what its offsets name), derived again here from the edge list
alone: adjacency, Kahn order, levels and places, the order by tie-break class, chains; and the object that lowers one class
after the other leaves the bytes that a fresh one does.  CPU only."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from tests.helpers import seeded_batch

HDR = ("n_nodes n_slots n_succ n_init n_groups n_gmembers off_node off_succ off_init off_topo off_slot off_group off_gmember "
       "off_pbeg off_pred n_levels off_lrec off_lbeg off_orec off_glvl off_place off_umap bytes structure split error id").split()
NODE = np.dtype([("succ_begin", "<u2"), ("n_succ", "u1"), ("slot", "u1"), ("ptkey", "u1"), ("blocked", "u1"), ("indeg", "u1"), ("cond", "u1")])
LEVEL = np.dtype([("succ", "<u2", 4), ("node", "<u2"), ("slot", "u1"), ("blocked", "u1"), ("cond", "u1"), ("indeg", "u1"), ("n_succ", "u1"), ("pad", "u1")])
ORDER = np.dtype([("at", "<u2"), ("b0", "<u2"), ("b1", "<u2"), ("chain_n", "u1"), ("chain_i", "u1")])


def check_blob(blob, edges):
    h = dict(zip(HDR, blob[:4 * len(HDR)].view("<u4").tolist()))
    n = h["n_nodes"]

    def at(off, dtype, count):
        size = np.dtype(dtype).itemsize * count
        assert h[off] + size <= h["bytes"] == len(blob)
        return blob[h[off]:h[off] + size].view(dtype)

    succ = [[] for _ in range(n)]
    pred = [[] for _ in range(n)]
    for a, b in edges:
        assert b not in succ[a]
        succ[a].append(int(b))
        pred[b].append(int(a))
    node = at("off_node", NODE, n)
    flat = at("off_succ", "<u2", h["n_succ"]).tolist()
    for v in range(n):
        b = int(node["succ_begin"][v])
        assert flat[b:b + int(node["n_succ"][v])] == succ[v] and node["indeg"][v] == len(pred[v])
    pbeg, p = at("off_pbeg", "<u2", n + 1).tolist(), at("off_pred", "<u2", len(edges)).tolist()
    assert [p[pbeg[v]:pbeg[v + 1]] for v in range(n)] == pred
    init = [v for v in range(n) if not pred[v]]
    assert at("off_init", "<u2", h["n_init"]).tolist() == init
    left, topo = [len(x) for x in pred], list(init)
    for v in topo:
        for w in succ[v]:
            left[w] -= 1
            if left[w] == 0:
                topo.append(w)
    assert at("off_topo", "<u2", n).tolist() == topo and h["error"] == 0
    # levels, and the nodes by (level, number)
    level = [0] * n
    for v in reversed(topo):
        level[v] = max([level[w] + 1 for w in succ[v]], default=0)
    assert h["n_levels"] == max(level) + 1
    by_level = sorted(range(n), key=lambda v: (level[v], v))
    place = [0] * n
    for k, v in enumerate(by_level):
        place[v] = k
    assert at("off_place", "<u2", n).tolist() == place
    assert at("off_lbeg", "<u2", h["n_levels"] + 1).tolist() == [sum(x < l for x in level) for l in range(h["n_levels"] + 1)]
    lrec = at("off_lrec", LEVEL, n)
    assert h["off_lrec"] % 16 == 0 and h["bytes"] % 16 == 0
    for k, v in enumerate(by_level):
        r = lrec[k]
        assert r["node"] == v and r["succ"].tolist() == ([place[w] for w in succ[v]] + [n] * 4)[:4]
        for f in ("slot", "blocked", "cond", "indeg", "n_succ"):
            assert r[f] == node[f][v], f
    # chains, and the nodes by (tie-break class, number)
    group = at("off_group", "<u2", 2 * h["n_groups"]).reshape(-1, 2).tolist()
    member, glvl = at("off_gmember", "<u2", h["n_gmembers"]).tolist(), at("off_glvl", "<u2", h["n_gmembers"]).tolist()
    assert glvl == [place[v] for v in member] and sum(c for _, c in group) == len(member)
    chain = {}
    for b, c in group:
        for j, v in enumerate(member[b:b + c]):
            assert v not in chain
            chain[v] = (c, j)
    orec, key = at("off_orec", ORDER, n), node["ptkey"].tolist()
    for k, v in enumerate(sorted(range(n), key=lambda v: (key[v], v))):
        r = orec[k]
        assert r["at"] == place[v] and (r["chain_n"], r["chain_i"]) == chain.get(v, (1, 0))
        assert r["b0"] == sum(x < key[v] for x in key) and r["b1"] == sum(x <= key[v] for x in key)
    # slots (some only of nodes that were taken out again), each with a place of its own in the universe
    assert max(node["slot"].tolist()) < h["n_slots"]
    umap = at("off_umap", "u1", h["n_slots"]).tolist()
    assert len(set(umap)) == len(umap)
    return n


@pytest.mark.parametrize("c,K", [(1, 4), (1, 12), (2, 4), (3, 4), (4, 1), (4, 16), (5, 4)])
def test_tables_of_a_class_follow_from_its_edges(c, K):
    cfg, batch = seeded_batch(c, 400)
    port = CpuPort(replace(cfg.problem, K_eval=K))
    sigs = np.unique(port.eval(batch)["sig"])
    sigs = sigs[sigs != np.uint64(2 ** 64 - 1)]
    sizes = set()
    for sig in sigs[:60]:
        blob, edges = port.blob(sig)
        again, edges2 = port.blob(sig, own=True)
        assert np.array_equal(blob, again) and np.array_equal(edges, edges2)
        sizes.add(check_blob(blob, edges))
    assert len(sizes) > 1 or len(sigs) == 1

