"""Bookkeeping of sets with many selections a step (a workgroup per set from 256
selections, in launches of many sets from 512): misses, slots, flags and LRU state bit-exact against the
oracle at run lengths around a wavefront's share, and the same errors."""
import numpy as np
import pytest
import torch

import ferry_amd as F

from test_gpu_parity import Pair, _zipf_stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group,k,n_req,cap", [
    (1, 255, 3, 300),    # the largest set of the one-wavefront kernel
    (1, 256, 3, 257),    # one wavefront's run each; almost every block evicted
    (1, 257, 2, 300),    # a run of one position
    (1, 256, 257, 270),  # 1028 sets: past four per CU, a wavefront per set again (256 CUs)
    (1, 512, 257, 520),  # ... and sets of 512 selections, which keep the workgroup
    (5, 57, 13, 320),    # 285 positions, the last group has 3 members
    (32, 40, 40, 1400),  # 1280 positions, the last group has 8 members
    (16, 64, 32, 1536),  # the shared-prefix shape
])
def test_group_bookkeeping_bit_exact(group, k, n_req, cap):
    mb, sels = _zipf_stream(n_req, 2, 2, k, 300, 400, 5, group=group, prefix=100 if group > 1 else 0,
                            seed=k)
    p = Pair(n_req, 2, 2, 4, k, cap, mb, F.FP8, group=group)
    rng = np.random.default_rng(k)
    for t, sel in enumerate(sels):
        sel = np.array(sel, np.uint32).reshape(-1)
        if t == 2:  # holes, and whole rows empty
            sel[rng.random(sel.size) < 0.3] = F.EMPTY
            sel.reshape(-1, k)[::5] = F.EMPTY
        p.check_fetched_bytes(p.step(sel))
        p.check_state()


def test_group_bookkeeping_errors():
    group, k, n_req = 8, 64, 8
    mb, sels = _zipf_stream(n_req, 1, 1, k, 600, 800, 1, group=1, seed=5)
    sel = np.array(sels[0], np.uint32).reshape(n_req, k)
    distinct = np.unique(sel).size
    assert distinct > 128
    for cap, bad_id, code in ((distinct - 1, None, -4), (distinct, mb, -3)):  # ECAPACITY, ERANGE
        ex = F.Executor(n_req, 1, 1, k, cap, mb, q_heads=2, group=group, dtype=F.F16, host_blocks=4099)
        bufs = ex.alloc_step_buffers()
        s = sel.copy()
        if bad_id is not None:
            s[3, 7] = bad_id
        ex.fetch_step(torch.from_numpy(s.view(np.int32)).cuda(), bufs)
        torch.cuda.synchronize()
        assert ex.stats()["device_error"] == code
        assert int(bufs["miss_count"].sum()) == 0
        fill, _, tag = ex.sets_state()
        assert np.all(fill == 0) and np.all(tag == 0xFFFFFFFF)
        ex.close()
    ex = F.Executor(n_req, 1, 1, k, distinct, mb, q_heads=2, group=group, dtype=F.F16, host_blocks=4099)
    bufs = ex.alloc_step_buffers()  # every slot of the set taken, none short
    ex.fetch_step(torch.from_numpy(sel.view(np.int32)).cuda(), bufs)
    torch.cuda.synchronize()
    assert ex.stats()["device_error"] == 0 and int(bufs["miss_count"].sum()) == distinct
