"""What the kernel of a few lanes per plan takes for granted of a chain -- its nodes are a run of the ids of one tie-break class, each
a successor of the one before -- is looked up when a class is lowered (rpeg_lower.h: chains_in_sequence); a class without it
has no ready-time rows and goes to the other kernels.  CPU only."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort, lib
from tests.helpers import seeded_batch
from tests.test_class_blob import HDR


def in_sequence(ptkey, succ, chains):
    key = np.array(ptkey, np.uint8)
    beg = np.cumsum([0] + [len(s) for s in succ]).astype(np.int32)
    to = np.array([v for s in succ for v in s] + [0], np.int32)
    cbeg = np.cumsum([0] + [len(c) for c in chains]).astype(np.int32)
    of = np.array([v for c in chains for v in c] + [0], np.int32)
    return bool(lib().port_chains_in_sequence(len(key), key.ctypes.data, beg.ctypes.data, to.ctypes.data, len(chains), cbeg.ctypes.data, of.ctypes.data))


@pytest.mark.parametrize("ptkey,succ,chains,want", [
    ([9, 9, 9], [[1], [2], []], [[0, 1, 2]], True),
    ([9, 9, 9], [[2, 1], [2], []], [[], [0, 1, 2], []], True),
    ([9, 4, 9, 4, 9], [[1, 2], [4], [3, 4], [], []], [[0, 2, 4]], True),        # nodes of another class between them
    ([9, 9, 9, 9], [[1], [], [3], []], [[0, 1], [2, 3]], True),
    ([9, 9, 9], [[2], [], []], [[0, 2]], False),                                # another node of the class between them
    ([9, 9, 9, 9], [[2], [3], [], []], [[0, 2], [1, 3]], False),                # two chains interleaved
    ([9, 9, 9], [[], [2], [0]], [[1, 2, 0]], False),                            # not by id
    ([9, 9, 9], [[1, 2], [], []], [[0, 1, 2]], False),                          # no edge from the second to the third
    ([9, 9, 8], [[1], [2], []], [[0, 1, 2]], False),                            # two classes
    ([9], [[]], [], True),
])
def test_chains_out_of_sequence_are_found(ptkey, succ, chains, want):
    assert in_sequence(ptkey, succ, chains) == want


@pytest.mark.parametrize("c,K", [(1, 4), (1, 12), (2, 4), (3, 6), (4, 1), (5, 4)])
def test_chains_of_the_workloads_are_in_sequence(c, K):
    cfg, batch = seeded_batch(c, 1500)
    port = CpuPort(replace(cfg.problem, K_eval=K))
    sigs = np.unique(port.eval(batch)["sig"])
    for sig in sigs[sigs != np.uint64(2 ** 64 - 1)]:
        blob, _ = port.blob(sig)
        n_nodes, n_rows = blob[:4 * (len(HDR) + 4)].view("<u4")[[HDR.index("n_nodes"), len(HDR)]]
        assert n_rows > 0 or n_nodes > 511
