"""Batches whose launches of the few-lanes-per-plan kernel are one, two or three, on the streams of a call that lays them out ahead and
of one that does not, timed and not: every stream waits for the layout before its first launch.  The oracle is the host build,
bit for bit.  (One launch: on the caller's stream.  Of two, the second on a stream of its own, of three the last two.)"""

import numpy as np
import pytest

from oracle.cpu_port import CpuPort
from rpeg_amd.engine import abi
from tests.helpers import seeded_batch
from tests.test_positions import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("c,n,most", [(4, 17000, 1), (5, 20011, 2), (2, 17000, 2), (3, 30000, 2), (2, 65536, 3), (1, 30000, 3)])
def test_launches_of_a_call(c, n, most):
    from rpeg_amd.engine.runtime import DeviceBatch, Engine
    cfg, batch = seeded_batch(c, n)
    want = CpuPort(cfg.problem).eval(batch, flags=abi.GATE_STALE, threads=16)
    eng = Engine(cfg.problem)
    resident, launches = DeviceBatch(batch, "cuda:0"), set()
    out = eng.alloc_outputs(batch.n)
    try:
        for side, timing in ((True, False), (True, True), (False, False), (False, True)):
            eng.set_side_layout(side)
            eng.set_timing(timing)
            for call in range(6):   # (24 entries first, then by what the plans had)
                eng.eval_device(resident, out, gate_stale=True)
                got = {k: v.cpu().numpy() for k, v in out.items()}
                s = eng.stats()
                assert s["side_layout"] == side
                if s["quad_tasks"]:
                    launches.add(s["quad_launches_8"] + s["quad_launches_16"] + s["quad_launches_24"])
                assert np.array_equal(got["mask"], want["mask"]), (side, timing, call)
                for k in ("makespan", "peak", "score"):
                    assert same_bits(got[k], want[k]), (k, side, timing, call)
                for v in out.values():
                    v.zero_()
            assert not timing or eng.last_kernel_ms() > 0.0
    finally:
        eng.close()
    assert launches and max(launches) == most, launches
