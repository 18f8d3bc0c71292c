"""Attention launches of few rows attend each row in parts, shared between
several workgroups that meet in per-stream memory, or one after the other in one
workgroup where there is none: parity with the oracle at the row counts where
the number of parts changes, on ragged and empty rows, infinite values as in
whole rows, and the same bits from concurrent streams, repeated launches and a
captured graph.  Rows whose weights are rounded to fp16 are always whole."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import ferry_amd as F
from oracle import pyoracle as O

from test_gpu_parity import TOL, Pair, _zipf_stream

pytestmark = pytest.mark.gpu


def _rel(a, b):
    den = np.maximum(np.abs(b).max(axis=-1), 1e-30)
    return (np.abs(a - b).max(axis=-1) / den).max()


@pytest.mark.parametrize("dtype,Hkv,Hq,n_req,k", [
    (F.F32, 1, 1, 1, 16),      # one row, 2 workgroups (256 CUs)
    (F.BF16, 2, 8, 4, 67),     # 8 rows, 8 workgroups, the wavefronts' shares uneven
    (F.BF16, 1, 8, 33, 33),    # 33 rows, 4 workgroups
    (F.FP8, 1, 8, 33, 33),     # 33 rows, 1 (fp16 weights)
    (F.F16, 2, 2, 43, 24),     # 86 rows, 2 (vector ALUs)
    (F.BF16, 2, 4, 64, 40),    # 128 rows, 2
    (F.F16, 2, 4, 64, 40),     # 128 rows, 1 (fp16 weights)
    (F.F32, 2, 4, 65, 50),     # 130 rows, 3
    (F.BF16, 2, 16, 85, 49),   # 170 rows, 3
    (F.F32, 2, 4, 65, 25),     # 130 rows, 1: thirds begin at 48 blocks
    (F.BF16, 2, 16, 8, 23),    # 16 rows, 1: parts begin at 24 blocks
    (F.BF16, 3, 6, 57, 30),    # 171 rows, 1
    (F.FP8, 3, 3, 57, 30),
])
def test_row_split_parity(dtype, Hkv, Hq, n_req, k):
    mb, sels = _zipf_stream(n_req, 1, Hkv, k, 80, 160, 1, seed=k)
    sel = np.array(sels[0], np.uint32).reshape(n_req, 1, Hkv, k).copy()
    for r in range(n_req):  # ragged rows: whole, one block, none, holes
        if r % 4 == 1:
            sel[r, :, :, 1:] = F.EMPTY
        elif r % 4 == 2:
            sel[r] = F.EMPTY
        elif r % 4 == 3:
            sel[r, :, :, ::3] = F.EMPTY
    p = Pair(n_req, 1, Hkv, Hq, k, 2 * k, mb, dtype)
    p.step(sel.reshape(-1))
    q = np.random.default_rng(k).standard_normal((n_req, 1, Hq, 128)).astype(np.float32)
    dq = torch.from_numpy(q).cuda()
    out, again = torch.full_like(dq, 7.0), torch.full_like(dq, -7.0)
    p.ex.sparse_decode(dq, p.bufs["slots"], out)
    p.ex.sparse_decode(dq, p.bufs["slots"], again)
    torch.cuda.synchronize()
    got = out.cpu().numpy().reshape(-1, 128).astype(np.float64)
    ref = O.attention_f64(p.g, sel.reshape(-1), q).reshape(-1, 128)
    none = np.repeat(np.all(sel == F.EMPTY, axis=-1).reshape(-1), Hq // Hkv)
    assert np.all(got[none] == 0.0)
    if not none.all():
        assert _rel(got[~none], ref[~none]) < TOL[dtype]
    assert torch.equal(out, again)  # parts are merged in part order
    assert p.ex.stats()["device_error"] == 0


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype,Hkv,Hq,k", [(F.F32, 2, 16, 160), (F.F16, 2, 2, 48), (F.BF16, 2, 8, 67),
                                             (F.BF16, 1, 8, 160)])
def test_rows_without_split_memory_give_the_same_bits(dtype, Hkv, Hq, k, waves, monkeypatch):
    """A context without memory for split rows attends them in one workgroup (the
    states of up to 8 parts of 8 heads in LDS) and selects from whole rows."""
    monkeypatch.setenv("FERRY_ATTN_WAVES", str(waves))
    n_req = 9
    mb, sels = _zipf_stream(n_req, 1, Hkv, k, 800, 900, 1, seed=k)
    q = torch.randn((n_req, 1, Hq, 128), device="cuda")
    ctx = torch.full((n_req,), mb, dtype=torch.int32, device="cuda")
    outs, picks = [], []
    for split in (1, 0):
        monkeypatch.setenv("FERRY_SPLIT", str(split))
        p = Pair(n_req, 1, Hkv, Hq, k, 2 * k, mb, dtype)
        p.step(sels[0])
        p.ex.summaries_build()
        outs.append(torch.full_like(q, 7.0))
        picks.append(torch.full((n_req, 1, Hkv, k), -7, dtype=torch.int32, device="cuda"))
        p.ex.sparse_decode(q, p.bufs["slots"], outs[-1])
        p.ex.select_topk(q, ctx, picks[-1])
        torch.cuda.synchronize()
        assert p.ex.stats()["device_error"] == 0
    assert torch.equal(outs[0], outs[1])
    assert torch.equal(picks[0], picks[1])


class _Pool:
    def __init__(self, ex):
        self.__cuda_array_interface__ = dict(shape=(ex.pool_slots, ex.block_bytes), typestr="|u1",
                                             version=2, data=(ex.pool_ptrs()[0], False))


def _whole_and_layered(dtype, Hkv, Hq, k, waves, monkeypatch, edit=None):
    """One executor's attention over 200 rows at once (whole rows) and layer by
    layer (10 rows: parts); edit(pool, slots) first changes stored values."""
    monkeypatch.setenv("FERRY_ATTN_WAVES", str(waves))
    n_req, L = 10 // Hkv, 20
    print(f"[row split] dtype={dtype} Hkv={Hkv} Hq={Hq} k={k} waves={waves}", flush=True)
    mb, sels = _zipf_stream(n_req, L, Hkv, k, 80, 160, 1, seed=k)
    p = Pair(n_req, L, Hkv, Hq, k, 2 * k, mb, dtype)
    p.step(sels[0])
    torch.cuda.synchronize()
    if edit:
        edit(torch.as_tensor(_Pool(p.ex), device="cuda"), p.bufs["slots"].view(n_req, L, Hkv, k))
    q = torch.randn((n_req, L, Hq, 128), device="cuda", generator=torch.Generator("cuda").manual_seed(k))
    whole, parts = torch.full_like(q, 7.0), torch.full_like(q, -7.0)
    p.ex.sparse_decode(q, p.bufs["slots"], whole)
    for l in range(L):
        p.ex.sparse_decode_layers(l, 1, q, p.bufs["slots"], parts)
    torch.cuda.synchronize()
    assert p.ex.attn_kernel()[1] == waves
    assert p.ex.stats()["device_error"] == 0
    return whole, parts


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype,Hkv,Hq", [(F.FP8, 2, 8), (F.FP8, 2, 2), (F.F16, 2, 4), (F.F16, 1, 8)])
def test_fp16_weights_do_not_depend_on_the_launch(dtype, Hkv, Hq, waves, monkeypatch):
    whole, layered = _whole_and_layered(dtype, Hkv, Hq, 48, waves, monkeypatch)
    assert torch.equal(whole, layered)


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("dtype,Hkv,Hq", [(F.F32, 1, 1), (F.F32, 2, 16), (F.F16, 2, 2), (F.BF16, 2, 2),
                                          (F.BF16, 2, 4), (F.BF16, 1, 8)])
def test_parts_differ_from_whole_rows_by_rounding_only(dtype, Hkv, Hq, waves, monkeypatch):
    # both within half the fp32 (or two-term bf16) tolerance of the 64-bit result
    whole, parts = _whole_and_layered(dtype, Hkv, Hq, 48, waves, monkeypatch)
    tol = 5e-5 if dtype == F.BF16 and Hq > Hkv else 1e-5
    assert _rel(parts.cpu().numpy(), whole.cpu().numpy()) < tol


@pytest.mark.parametrize("pos", [0, 1, 39])
@pytest.mark.parametrize("dtype,Hkv,Hq,np_dtype", [(F.F32, 1, 2, torch.float32), (F.F16, 2, 2, torch.float16),
                                                   (F.BF16, 2, 8, torch.bfloat16)])
def test_infinite_values_in_parts_are_those_of_whole_rows(dtype, Hkv, Hq, np_dtype, pos, monkeypatch):
    """40 blocks in 5 parts of 4 wavefronts: blocks 0 and 1 are in the first part,
    39 in the last.  Infinities and NaN come out where a whole row has them, and
    nowhere else."""
    def edit(pool, slots):
        for l in range(slots.shape[1]):
            for r in range(slots.shape[0]):
                v = pool[int(slots[r, l, 0, pos])].view(np_dtype).view(2, 16, 128)[1]
                v[r % 16, 5] = float("inf")
                v[3, 77] = -float("inf")

    whole, parts = _whole_and_layered(dtype, Hkv, Hq, 40, 4, monkeypatch, edit)
    hit = (~torch.isfinite(whole)).any()
    assert bool(hit)
    assert torch.equal(torch.isnan(whole), torch.isnan(parts))
    assert torch.equal(torch.isinf(whole), torch.isinf(parts))
    inf = torch.isinf(whole)
    assert torch.equal(whole[inf], parts[inf])
    if dtype != F.BF16:  # a bf16 weight's second term may be 0
        assert bool(inf.any()) and not bool(torch.isnan(whole).any())
    fin = torch.isfinite(whole)
    assert float((whole - parts)[fin].abs().max()) < 1e-4


def test_row_split_streams_and_graphs():
    """Six streams at once on one context (not all have split state), each with
    queries and outputs of its own, then with the same queries, and a graph
    captured from one of them replayed between eager launches: the same bits
    from all of them."""
    n_req, Hkv, Hq, k = 8, 2, 8, 64
    mb, sels = _zipf_stream(n_req, 1, Hkv, k, 80, 160, 1, seed=3)
    p = Pair(n_req, 1, Hkv, Hq, k, 2 * k, mb, F.BF16)
    p.step(sels[0])
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(6)]
    qs = [torch.randn((n_req, 1, Hq, 128), device="cuda") for _ in streams]
    outs = [torch.zeros_like(q) for q in qs]
    torch.cuda.synchronize()
    for _ in range(20):
        for s, q, o in zip(streams, qs, outs):
            p.ex.sparse_decode(q, p.bufs["slots"], o, stream=s)
    torch.cuda.synchronize()
    refs = [O.attention_f64(p.g, sels[0], q.cpu().numpy()).reshape(-1, 128) for q in qs]
    for o, ref in zip(outs, refs):
        assert _rel(o.cpu().numpy().reshape(-1, 128), ref) < TOL[F.BF16]
    first = outs[0].clone()
    torch.cuda.synchronize()
    for s, o in zip(streams, outs):
        p.ex.sparse_decode(qs[0], p.bufs["slots"], o, stream=s)
    torch.cuda.synchronize()
    for o in outs:
        assert torch.equal(o, first)
    second = torch.empty_like(first)
    p.ex.sparse_decode(qs[1], p.bufs["slots"], second)
    g = torch.cuda.CUDAGraph()
    gout = torch.zeros_like(qs[1])
    with torch.cuda.graph(g, stream=streams[0]):
        p.ex.sparse_decode(qs[1], p.bufs["slots"], gout, stream=streams[0])
    for _ in range(3):
        gout.zero_()
        outs[0].zero_()
        torch.cuda.synchronize()
        g.replay()
        p.ex.sparse_decode(qs[0], p.bufs["slots"], outs[0], stream=streams[0])
        torch.cuda.synchronize()
        assert torch.equal(gout, second)
        assert torch.equal(outs[0], first)
    assert p.ex.stats()["device_error"] == 0


@pytest.mark.parametrize("dtype,Hq", [(F.F32, 2), (F.BF16, 8), (F.FP8, 8)])
def test_adaptive_steps_do_not_depend_on_their_ranges(dtype, Hq):
    """The same steps in one layer range and in eight: the same bits, though a
    range of few rows is a launch of few rows."""
    n_req, L, Hkv, k = 4, 8, 2, 48
    mb, sels = _zipf_stream(n_req, L, Hkv, k, 200, 300, 4, seed=9)
    pairs = [Pair(n_req, L, Hkv, Hq, k, 2 * k, mb, dtype) for _ in range(2)]
    pairs[0].ex.set_batch_policy(512.0, 512.0, 1.0)
    pairs[1].ex.set_batch_policy(1e-3, 1e-3, 1.0)
    assert pairs[0].ex.decode_chunks(100) == 1 and pairs[1].ex.decode_chunks(100) == L
    side = torch.cuda.Stream()
    for sel in sels:
        ds = torch.from_numpy(np.array(sel, np.uint32).view(np.int32)).cuda().view(n_req, L, Hkv, k)
        q = torch.randn((n_req, L, Hq, 128), device="cuda")
        outs = []
        for p in pairs:
            out = torch.full_like(q, 7.0)
            p.ex.decode_step(ds, q, p.bufs, out, side_stream=side)
            torch.cuda.synchronize()  # the next step knows what this one fetched
            assert p.ex.stats()["device_error"] == 0
            outs.append(out)
        assert torch.equal(outs[0], outs[1])


class _Streams:
    """Streams created and destroyed through the HIP runtime (torch keeps its own)."""

    def __init__(self):
        self.hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime already loaded with torch

    def create(self):
        h = ctypes.c_void_p()
        assert self.hip.hipStreamCreate(ctypes.byref(h)) == 0
        return torch.cuda.ExternalStream(h.value)

    def destroy(self, s):
        assert self.hip.hipStreamDestroy(ctypes.c_void_p(s.cuda_stream)) == 0


def _few_rows(k=128, seed=3):
    n_req, Hkv, Hq = 4, 2, 8
    mb, sels = _zipf_stream(n_req, 1, Hkv, k, 200, 400, 1, seed=seed)
    p = Pair(n_req, 1, Hkv, Hq, k, 2 * k, mb, F.BF16)
    p.step(sels[0])
    qs = [torch.randn((n_req, 1, Hq, 128), device="cuda") for _ in range(8)]
    want = [torch.empty_like(q) for q in qs]
    for q, w in zip(qs, want):
        p.ex.sparse_decode(q, p.bufs["slots"], w)
    torch.cuda.synchronize()
    return p, qs, want


def test_streams_that_come_and_go():
    """Streams destroyed behind queued launches, whose handles new streams may
    get: the same bits from all.  Split state goes back to later streams: the
    last of twenty is as fast as the first."""
    p, qs, want = _few_rows()
    st = _Streams()
    outs = [torch.zeros_like(qs[0]) for _ in range(40)]
    torch.cuda.synchronize()
    for i in range(40):
        s = st.create()
        with torch.cuda.stream(s):
            torch.cuda._sleep(200_000)
        for _ in range(3):
            p.ex.sparse_decode(qs[i % 8], p.bufs["slots"], outs[i], stream=s)
        st.destroy(s)
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        assert torch.equal(o, want[i % 8]), i
    us = []
    for i in range(20):
        s = st.create()
        best = float("inf")
        for _ in range(3):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            with torch.cuda.stream(s):
                torch.cuda._sleep(4_000_000)
            a.record(s)
            for _ in range(64):
                p.ex.sparse_decode(qs[0], p.bufs["slots"], outs[0], stream=s)
            b.record(s)
            s.synchronize()
            best = min(best, a.elapsed_time(b) / 64e-3)
        us.append(best)
        st.destroy(s)
    print("[row split] us per launch on 20 streams:", [round(x, 1) for x in us], flush=True)
    assert max(us[4:]) < 1.6 * min(us[:3])  # one workgroup per row takes 3 times as long
    assert p.ex.stats()["device_error"] == 0


@pytest.mark.parametrize("shared", [False, True])
def test_host_threads_on_one_context(shared):
    """Four host threads launch on one context, each on a stream of its own or
    all on one."""
    p, qs, want = _few_rows(k=64, seed=5)
    one = torch.cuda.Stream()
    errors = []

    def work(t):
        try:
            s = one if shared else torch.cuda.Stream()
            outs = [torch.zeros_like(q) for q in qs]
            torch.cuda.synchronize()
            for _ in range(50):
                for i in range(t, t + 4):
                    p.ex.sparse_decode(qs[i % 8], p.bufs["slots"], outs[i % 8], stream=s)
            s.synchronize()
            for i in range(t, t + 4):
                assert torch.equal(outs[i % 8], want[i % 8]), (t, i)
        except BaseException as e:  # reported by the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert p.ex.stats()["device_error"] == 0
