"""Start times as large as doubles get, in the kernel of a few lanes per plan: a slot without an entry has 0x7FEFFFFF in the high word
of its time, so a plan with a start time from there on is flagged and redone by the launch that ends the call, and one whose
start times are all below it is not.  The oracle is the host build, bit for bit."""

from dataclasses import replace

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import oracle_eval, seeded_batch
from tests.test_positions import FREE_LINKS, same_bits

PLANS, COPIES = 24, 8


def high_word(x):
    return int(np.float64(x).view(np.uint64) >> np.uint64(32))


def problem(c, K, word):
    """(problem, plans, the one that starts last) with a last start time of all plans of that high word: operators alone take time,
    and all of them that much longer."""
    cfg, batch = seeded_batch(c, PLANS)
    p = replace(cfg.problem, K_eval=K, hw=replace(cfg.problem.hw, **FREE_LINKS))
    last = [max(oracle_eval(p, batch, i, want_trace=True)["start"].values()) for i in range(PLANS)]
    longer = float(np.uint64((word << 32) + (1 << 31)).view(np.float64)) / max(last)
    p = replace(p, hw=replace(p.hw, op_generation_scale=longer, op_inference_scale=longer, op_training_scale=longer))
    return p, batch, int(np.argmax(last))


CASES = [(1, 4), (2, 5), (3, 2), (4, 12), (5, 3)]


@pytest.mark.parametrize("c,K", CASES)
@pytest.mark.parametrize("word", [0x7FEFFFFE, 0x7FEFFFFF])
def test_such_plans_exist(c, K, word):
    p, batch, latest = problem(c, K, word)
    last = [max(oracle_eval(p, batch, i, want_trace=True)["start"].values()) for i in range(PLANS)]
    assert high_word(last[latest]) == word == high_word(max(last)) and sum(high_word(x) == word for x in last) < PLANS / 2
    out = CpuPort(p).eval(batch)
    assert (out["mask"] & abi.MASK_VALID != 0).all() and (out["mask"] & abi.MASK_ERROR == 0).all()
    assert np.isinf(out["makespan"][latest]) and np.isfinite(out["makespan"]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("c,K", CASES)
def test_start_times_below_the_word_of_empty_slots_and_at_it(c, K):
    from rpeg_amd.engine.runtime import Engine
    redone = {}
    for word in (0x7FEFFFFE, 0x7FEFFFFF):
        p, batch, latest = problem(c, K, word)
        batch = batch.take(np.tile(np.arange(PLANS), COPIES))
        want = CpuPort(p).eval(batch, flags=abi.GATE_STALE, threads=16)
        eng = Engine(p)
        eng.set_state_lanes(4)
        try:
            for call in range(4):   # (24 entries first, then by what the plans had)
                out = eng.eval(batch, gate_stale=True)
                s = eng.stats()
                assert s["quad_plans"] == batch.n
                redone[word] = s["redone_before"]     # (of the call before)
                assert np.array_equal(out["mask"], want["mask"]), (word, call)
                for k in ("makespan", "peak", "score"):
                    assert same_bits(out[k], want[k]), (word, call, k)
        finally:
            eng.close()
    assert redone[0x7FEFFFFF] >= redone[0x7FEFFFFE] + COPIES, redone
