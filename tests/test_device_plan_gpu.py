"""Decode calls without host lengths: the kernels plan the context splits from
the device lengths (one captured call serves every step of growing sequences).
Against the oracle at batch sizes around a wave's 64 lanes, ragged and empty
sequences and lengths around the split sizes, with the workspace between guard
bands; and with a workspace of the static plan's size, which keeps that plan."""
import ctypes

import numpy as np
import pytest
import torch

from mugen_amd import _capi
from mugen_amd import attention as A
from tests import cases as C
from tests.test_bounds_gpu import Guarded, guarded_ws
from tests.test_kv_q4_gpu import build_store, oracle_decode

pytestmark = pytest.mark.gpu


def lens_of(B, hi, seed):
    x = np.random.default_rng(seed).integers(0, hi + 1, B).astype(np.int32)
    x[0] = hi
    if B > 2:
        x[1], x[B - 1] = 0, 1
    return x


def planned(ws, size, per, bound):
    """The chunk that the call left for its merge, after the partials of as many
    splits (`per` bytes each, at most `bound`) as the workspace holds; None when
    the call kept the static plan (the workspace was filled with 0xff)."""
    fit = min((size - 512) // per, bound)
    chunk = int(ws.t[fit * per:fit * per + 4].cpu().numpy().view(np.int32)[0])
    return None if chunk == -1 else chunk


def check_planned(chunk, on_device=True):
    if on_device:
        assert chunk is not None and chunk > 0 and chunk % 32 == 0, f"the device plan is taken: {chunk}"
    else:
        assert chunk is None, f"the static plan stays: {chunk}"


# one guess up to 4 and up to 8 sequences, a search above, past the wave's 64
# lanes, head_dim 256 (half the round), padded heads; then caches whose static plan
# has chunks of 128 tokens or less, or of 256 for a few sequences, which stays
@pytest.mark.parametrize("B,H,Hk,D,hi,cache,on_device", [
    (1, 8, 8, 64, 700, 8192, True), (1, 7, 1, 128, 1, 6000, True), (1, 16, 16, 64, 6000, 6000, True),
    (4, 32, 32, 64, 777, 2048, True), (8, 16, 16, 64, 900, 1024, True), (5, 28, 4, 128, 1500, 4096, True),
    (16, 16, 4, 128, 300, 2048, True), (64, 4, 4, 64, 400, 512, True), (65, 3, 1, 64, 500, 2048, True),
    (127, 2, 2, 64, 130, 1024, True), (3, 8, 2, 256, 900, 8192, True), (16, 8, 8, 256, 400, 512, True),
    (2, 4, 2, 96, 64, 8192, True), (7, 8, 4, 40, 1000, 4096, True), (32, 8, 8, 64, 2048, 2048, True),
    (16, 8, 8, 256, 1024, 1024, True),
    (16, 16, 4, 128, 300, 1024, False), (65, 3, 1, 64, 500, 640, False), (127, 2, 2, 64, 130, 256, False),
    (3, 8, 2, 256, 900, 2048, False), (2, 4, 2, 96, 64, 65, False), (4, 8, 8, 64, 900, 4096, False),
])
def test_gqa_plan_on_device(device, B, H, Hk, D, hi, cache, on_device):
    lens = lens_of(B, hi, B + hi)
    c = C.gqa_decode_case(2100 + B, B, H, Hk, D, lens, max_T=cache, dtype=C.F16)
    ref = C.gqa_decode_ref(c, nthreads=16)
    q, k, v = (C.to_dev(c[x], C.F16, device) for x in ("qb", "kb", "vb"))
    sl = torch.from_numpy(lens).to(device)
    C.say(f"gqa_decode without host lengths B={B} Hk={Hk} D={D} lens<={hi} cache={cache}")
    out = Guarded((B, H, D), torch.float32, device)
    L = _capi.lib()
    a = A.gqa_decode_args(q, k, v, sl, out.t, cache)
    need = L.mugen_attn_gqa_decode_workspace_size(ctypes.byref(a))
    host = np.full(B, cache, np.int32)  # every sequence full: the plan for max_seq_len
    a.seq_lens_host = host.ctypes.data
    static = L.mugen_attn_gqa_decode_workspace_size(ctypes.byref(a))
    a.seq_lens_host = None
    padded = 64 if D <= 64 else 128 if D <= 128 else 256
    for size in (need, static):
        ws = guarded_ws(size, device)
        ws.t.fill_(255)
        out.t.zero_()
        _capi.check(L.mugen_attn_gqa_decode(ctypes.byref(a), ctypes.c_void_p(ws.t.data_ptr()) if size else None, size,
                                            A._stream(device)))
        assert out.intact() and ws.intact(), "guard band overwritten"
        C.assert_close(out.t.cpu().numpy(), ref, f"gqa plan on device, workspace {size}")
        if size == need:
            check_planned(planned(ws, need, B * H * (padded * 4 + 8), min(32, -(-cache // 64))), on_device)


@pytest.mark.parametrize("B,H,q_len,hi,cache,on_device", [
    (1, 16, 1, 1000, 8192, True), (4, 128, 1, 3000, 8192, True), (8, 128, 1, 700, 8192, True),
    (5, 128, 1, 6000, 6000, True), (3, 128, 5, 600, 4096, True), (7, 16, 3, 500, 8192, True),
    (64, 16, 1, 90, 1024, True), (65, 16, 1, 70, 1024, True), (33, 128, 1, 200, 1024, True), (2, 16, 16, 333, 8192, True),
    (8, 128, 1, 700, 2048, False), (3, 128, 5, 600, 1024, False), (64, 16, 1, 90, 128, False),
    (65, 16, 1, 70, 96, False), (2, 16, 16, 333, 4096, False)])
def test_mla_plan_on_device(device, B, H, q_len, hi, cache, on_device):
    lens = np.maximum(lens_of(B, hi, B + hi), 0 if q_len == 1 else q_len).astype(np.int32)
    c = C.mla_case(2200 + B, B, q_len, H, lens, max_T=cache, q_dtype=C.F32, lat_dtype=C.F16)
    ref = C.mla_ref(c, nthreads=16)
    q, lat = C.to_dev(c["q"], C.F32, device), C.to_dev(c["latb"], C.F16, device)
    sl = torch.from_numpy(lens).to(device)
    C.say(f"mla_decode without host lengths B={B} H={H} q_len={q_len} lens<={hi} cache={cache}")
    out = Guarded((B, q_len, H, 512), torch.float32, device)
    L = _capi.lib()
    a = A.mla_args(q, lat, sl, out.t, cache, C.MLA_SCALE)
    need = L.mugen_attn_mla_decode_workspace_size(ctypes.byref(a))
    host = np.full(B, cache, np.int32)
    a.seq_lens_host = host.ctypes.data
    static = L.mugen_attn_mla_decode_workspace_size(ctypes.byref(a))
    a.seq_lens_host = None
    R = q_len * H
    for size in (need, static):
        ws = guarded_ws(size, device)
        ws.t.fill_(255)
        out.t.zero_()
        _capi.check(L.mugen_attn_mla_decode(ctypes.byref(a), ctypes.c_void_p(ws.t.data_ptr()), size, A._stream(device)))
        assert out.intact() and ws.intact(), "guard band overwritten"
        C.assert_close(out.t.cpu().numpy(), ref, f"mla plan on device, workspace {size}")
        if size == need:
            check_planned(planned(ws, need, B * ((R + 15) // 16 * 16 * 1024 + R * 8), min(32, -(-cache // 32))), on_device)


# the store rounds a sequence's Q4 and f16 tokens up to splits on their own: batches
# whose work lists come closest to the launch's workgroups (equal lengths, half a
# round of (sequence, kv head) pairs), each way to the plan.  A workspace of NaNs
# shows a work item that nobody took
@pytest.mark.parametrize("H,Hk,D,lens,keep,cache", [
    (8, 8, 64, [4600, 5853, 3424, 4723, 5733, 5020, 4463, 3623], 256, 8192),
    (16, 8, 64, [6100] * 4, 256, 8192),
    (8, 8, 64, [5000] * 6, 256, 8192),
    (16, 16, 64, [7168] * 2, 256, 8192),
    (16, 8, 128, [2900], 100, 8192),
    (2, 2, 256, [8000, 1, 0, 1024, 1024, 1024, 1024], 256, 8192),
    (16, 16, 64, [1000 + 37 * i for i in range(16)], 200, 2048),
    (4, 2, 64, [(131 * i) % 700 for i in range(66)], 32, 2048),
])
def test_q4_plan_on_device(device, H, Hk, D, lens, keep, cache):
    B, T, ring = len(lens), max(lens), 256
    nq = np.maximum(np.array(lens) - keep, 0).astype(np.int32)
    rng = np.random.default_rng(2300 + B)
    k, v, q = (rng.standard_normal(s, dtype=np.float32).astype(np.float16).view(np.uint16)
               for s in ((B, T, Hk * D), (B, T, Hk * D), (B, H, D)))
    store = build_store(k, v, lens, nq, ring, device)
    for i in (0, 1):  # the Q4 rows as the first of a cache's
        rows, store[i] = store[i], torch.zeros((B, cache, store[i].shape[2]), dtype=torch.uint8, device=device)
        store[i][:, :T] = rows
    qd, sl, nqd = C.to_dev(q, C.F16, device), torch.tensor(lens, dtype=torch.int32, device=device), torch.from_numpy(nq).to(device)
    out = Guarded((B, H, D), torch.float32, device)
    a = _capi.GqaDecodeQ4Args()
    a.store.q4_k, a.store.q4_v, a.store.ring_k, a.store.ring_v = [t.data_ptr() for t in store]
    a.store.q4_seq_stride, a.store.ring_seq_stride = store[0][0].numel(), store[2][0].numel()
    a.store.ring, a.store.fp16_preserve_last = ring, keep
    a.q, a.seq_lens, a.n_q4, a.out = qd.data_ptr(), sl.data_ptr(), nqd.data_ptr(), out.t.data_ptr()
    a.batch, a.n_heads, a.n_kv_heads, a.head_dim, a.max_seq_len, a.out_dtype = B, H, Hk, D, cache, C.F32
    L = _capi.lib()
    need = L.mugen_attn_gqa_decode_q4_workspace_size(ctypes.byref(a))
    ws = guarded_ws(need, device)
    ws.t.fill_(255)
    C.say(f"gqa_decode_q4 without host lengths B={B} Hk={Hk} D={D} lens<={T} cache={cache}")
    _capi.check(L.mugen_attn_gqa_decode_q4(ctypes.byref(a), ctypes.c_void_p(ws.t.data_ptr()), need, A._stream(device)))
    assert out.intact() and ws.intact(), "guard band overwritten"
    check_planned(planned(ws, need, B * H * (D * 4 + 8), min(32, -(-cache // 64)) + 1))
    C.assert_close(out.t.cpu().numpy(), oracle_decode(q, k, v, lens, nq, H, Hk, D), f"q4 plan on device B={B}")


def test_gqa_deep_plan(device):
    # a large ragged batch with host lengths: 1024-token items over several
    # rounds; without their workspace the call keeps one split per sequence
    B, H, Hk, D, cache = 64, 8, 8, 64, 2600
    lens = lens_of(B, cache, 77)
    c = C.gqa_decode_case(2400, B, H, Hk, D, lens, max_T=cache, dtype=C.F16)
    ref = C.gqa_decode_ref(c, nthreads=16)
    q, k, v = (C.to_dev(c[x], C.F16, device) for x in ("qb", "kb", "vb"))
    sl = torch.from_numpy(lens).to(device)
    C.say("gqa_decode deep plan")
    for with_ws in (True, False):
        out = Guarded((B, H, D), torch.float32, device)
        a = A.gqa_decode_args(q, k, v, sl, out.t, cache)
        a.seq_lens_host = lens.ctypes.data
        L = _capi.lib()
        need = L.mugen_attn_gqa_decode_workspace_size(ctypes.byref(a))
        assert (need - 256) // (B * H * (4 * D + 8)) == 3  # 2600 tokens in 1024s
        ws = guarded_ws(need, device)
        _capi.check(L.mugen_attn_gqa_decode(ctypes.byref(a), ctypes.c_void_p(ws.t.data_ptr()) if with_ws else None,
                                            need if with_ws else 0, A._stream(device)))
        assert out.intact() and ws.intact(), "guard band overwritten"
        C.assert_close(out.t.cpu().numpy(), ref, f"deep plan, workspace {with_ws}")


def test_gqa_deep_plan_sizes():
    # equal lengths stay in one round, unsplit (no workspace)
    a = _capi.GqaDecodeArgs()
    a.q = a.k_cache = a.v_cache = a.seq_lens = a.out = 0x1000
    a.batch, a.n_heads, a.n_kv_heads, a.head_dim, a.max_seq_len = 64, 32, 8, 128, 8192
    a.seq_stride, a.kv_dtype, a.out_dtype = 8192 * 8 * 128, C.F16, C.F16
    size = _capi.lib().mugen_attn_gqa_decode_workspace_size
    same = np.full(64, 8191, np.int32)
    a.seq_lens_host = same.ctypes.data
    assert size(ctypes.byref(a)) == 0
    ragged = np.linspace(512, 8191, 64).astype(np.int32)
    a.seq_lens_host = ragged.ctypes.data
    assert (size(ctypes.byref(a)) - 256) // (64 * 32 * (4 * 128 + 8)) == 8
