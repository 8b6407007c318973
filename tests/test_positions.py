"""Positions of the nodes in the order that breaks ties, in the kernels that schedule a plan with a wavefront or with a few
lanes: equal ranks counted along (small graphs) or afterwards, ranks of all, half or a quarter of a wavefront's plans at a
time, classes of one node to many per lane.  Links without latency make a transfer's rank that of the node behind it, so that
nodes of one tie-break class share positions by the dozen.  The oracle is the host build, bit for bit."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch

FREE_LINKS = {f"alpha_{k}_{t}": 0.0 for k in ("coll", "p2p") for t in "gnr"} | {f"beta_{k}_{t}": 0.0 for k in ("coll", "p2p") for t in "gnr"}


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float64).view(np.uint64), np.asarray(b, np.float64).view(np.uint64))


@pytest.mark.parametrize("c,K", [(1, 4), (2, 4), (3, 8), (5, 4)])
def test_nodes_of_a_chain_follow_each_other(c, K):
    """... in the order by tie-break class, joined by edges: the first one has the largest rank."""
    from tests.test_class_blob import HDR, ORDER
    cfg, batch = seeded_batch(c, 300)
    port = CpuPort(replace(cfg.problem, K_eval=K))
    sigs = np.unique(port.eval(batch)["sig"])
    chains = 0
    for sig in sigs[sigs != np.uint64(2 ** 64 - 1)][:40]:
        blob, edges = port.blob(sig)
        h = dict(zip(HDR, blob[:4 * len(HDR)].view("<u4").tolist()))
        n = h["n_nodes"]
        orec = blob[h["off_orec"]:h["off_orec"] + 8 * n].view(ORDER)
        place = blob[h["off_place"]:h["off_place"] + 2 * n].view("<u2").tolist()
        node = {p: v for v, p in enumerate(place)}
        edge = {(int(a), int(b)) for a, b in edges}
        group = blob[h["off_group"]:h["off_group"] + 4 * h["n_groups"]].view("<u2").reshape(-1, 2).tolist()
        member = blob[h["off_gmember"]:h["off_gmember"] + 2 * h["n_gmembers"]].view("<u2").tolist()
        at = {int(r["at"]): i for i, r in enumerate(orec)}
        for b, m in group:
            ids = [at[place[v]] for v in member[b:b + m]]
            assert ids == list(range(ids[0], ids[0] + m)) and [int(orec[i]["chain_i"]) for i in ids] == list(range(m))
            nodes = [node[int(orec[i]["at"])] for i in ids]
            assert all((nodes[j], nodes[j + 1]) in edge for j in range(m - 1))
            chains += 1
    assert chains or c == 4


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("c,K,n,free", [(2, 4, 700, False), (2, 5, 40000, False), (4, 16, 3000, True), (4, 2, 60000, True),
                                        (1, 3, 2000, True), (3, 4, 6000, True), (3, 8, 700, True), (5, 4, 16000, True)])
def test_positions_with_and_without_equal_ranks(c, K, n, free, lanes):
    from rpeg_amd.engine.runtime import Engine
    cfg, batch = seeded_batch(c, n)
    p = replace(cfg.problem, K_eval=K)
    if free:
        p = replace(p, hw=replace(p.hw, **FREE_LINKS))
    want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16, want_mass=n < 10000)
    eng = Engine(p)
    eng.set_state_lanes(lanes)
    try:
        for call in range(4):   # (k_quad: 24 entries first, then by what the plans had)
            mass = call == 3 and n < 10000
            out = eng.eval(batch, gate_stale=True, mass=mass)
            assert np.array_equal(out["mask"], want["mask"])
            for k in ("makespan", "peak", "score") + (("mass",) if mass else ()):
                assert same_bits(out[k], want[k]), (k, call)
    finally:
        eng.close()
