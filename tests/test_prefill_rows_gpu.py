"""Prefill over flattened (token, head) rows: 128-row blocks whose edges fall
anywhere in a token's heads, 32-key tiles in a 5-slot ring, key ranges with
their own partials.  Against the CPU oracle's flash_prefill_attention
restatement at the sizes where each can go wrong."""
import ctypes

import numpy as np
import pytest
import torch

import mugen_amd
from mugen_amd import _capi
from mugen_amd import attention as A
from tests import cases as C
from tests.test_bounds_gpu import Guarded, guarded_ws

pytestmark = pytest.mark.gpu


def run(c, device, out_dtype=C.F32, causal=True):
    """The call with its workspace and output between guard bands."""
    C.say(f"prefill rows N={c['N']} H={c['H']} Hk={c['Hk']} D={c['D']} start={c['start']} dtype={c['dtype']} "
          f"out={out_dtype} causal={causal}")
    q, k, v = (C.to_dev(c[x], c["dtype"], device) for x in ("qb", "kb", "vb"))
    out = Guarded((c["N"], c["H"], c["D"]), C.torch_dtype(out_dtype), device)
    a = A._prefill_args(q, k, v, c["start"], causal, out.t)
    need = _capi.lib().mugen_attn_gqa_prefill_workspace_size(ctypes.byref(a))
    ws = guarded_ws(need, device)
    mugen_amd.flash_prefill_attention(q, k, v, c["start"], causal=causal, out=out.t,
                                      workspace=ws.t if need else ws.t[:0])
    assert out.intact() and ws.intact(), "guard band overwritten"
    return out.t.float().cpu().numpy(), need


def check(c, device, what, out_dtype=C.F32):
    got, need = run(c, device, out_dtype)
    C.assert_close(got, C.prefill_ref(c, nthreads=16), what)
    return need


# one row past a block; blocks that end inside a token's heads (7 and 3 heads
# per kv head); one head per kv head; every deal of kv heads to the XCDs (1, 2,
# 3, 4, 8, 16); key counts around the tile and the ring; 16 heads per kv head
WIDE = [(129, 8, 8, 256, 0), (65, 16, 8, 256, 0), (150, 21, 3, 256, 0), (90, 12, 4, 256, 31), (300, 2, 1, 256, 1),
        (140, 32, 16, 136, 0), (130, 32, 2, 256, 32), (257, 6, 2, 200, 63), (160, 4, 2, 256, 0)]


@pytest.mark.parametrize("N,H,Hk,D,start", WIDE)
@pytest.mark.parametrize("dtype", [C.F16, C.BF16])
def test_wide_rows(device, N, H, Hk, D, start, dtype):
    check(C.prefill_case(1200 + N + D, N, H, Hk, D, start, dtype), device, f"rows N={N} D={D} Hk={Hk}")


# key ranges at head_dim above 128 (fp32 partials): the last range partial, a
# block whose rows end inside a range, and a single token
@pytest.mark.parametrize("N,H,Hk,D,start", [(5, 16, 8, 256, 1501), (1, 8, 2, 192, 2000), (140, 4, 1, 256, 1000),
                                            (33, 14, 2, 248, 900)])
@pytest.mark.parametrize("dtype", [C.F16, C.BF16])
def test_wide_rows_split(device, N, H, Hk, D, start, dtype):
    c = C.prefill_case(1300 + N + D, N, H, Hk, D, start, dtype)
    assert check(c, device, f"split rows N={N} D={D} start={start}") > 0, "the planner splits this chunk's keys"
    check(c, device, f"split rows N={N} D={D} start={start}, 16-bit output", dtype)


# head_dim up to 128: just past the workgroup counts where this kernel takes
# over (256, 320, 512, 640: prefill_rows_default), with and without the fp16
# copy of V.  The first rows, a stretch in the middle
# and the last rows, through the oracle's start-offset form
NARROW = [(2926, 28, 4, 128, 0), (1640, 40, 10, 96, 0), (1030, 32, 32, 128, 0), (1900, 33, 11, 64, 5), (2500, 33, 11, 64, 5),
          (3300, 16, 8, 64, 0), (860, 96, 16, 48, 3)]


@pytest.mark.parametrize("N,H,Hk,D,start", NARROW)
@pytest.mark.parametrize("dtype", [C.F16, C.BF16])
def test_narrow_rows(device, N, H, Hk, D, start, dtype):
    c = C.prefill_case(1600 + N + D, N, H, Hk, D, start, dtype)
    for passes in (0, 1) if dtype == C.BF16 else (0,):
        if passes == 0:
            got, _ = run(c, device)
        else:  # no workspace: V converted on chip
            q, k, v = (C.to_dev(c[x], dtype, device) for x in ("qb", "kb", "vb"))
            got = mugen_amd.flash_prefill_attention(q, k, v, start, out_dtype=torch.float32,
                                                    workspace=torch.empty(0, dtype=torch.uint8, device=device))
            got = got.cpu().numpy()
        for lo, n in ((0, 40), (N // 2 - 20, 40), (N - 40, 40)):
            kv = start + lo + n
            ref = C.O.gqa_prefill(c["q"][lo:lo + n], c["k"][:kv], c["v"][:kv], n, H, Hk, D, kv, start + lo, nthreads=16)
            C.assert_close(got[lo:lo + n], ref, f"rows N={N} D={D} rows {lo}..{lo + n}")


def test_wide_rows_not_causal(device):
    c = C.prefill_case(1400, 140, 8, 4, 256, 53, C.F16)
    got, _ = run(c, device, causal=False)
    N, H, Hk, D, kv = 140, 8, 4, 256, c["kv_len"]
    ref = C.O.gqa_attention(c["q"], c["k"].reshape(1, kv, Hk, D).repeat(N, 0), c["v"].reshape(1, kv, Hk, D).repeat(N, 0),
                            [kv] * N, H, Hk, D, kv * Hk * D)
    C.assert_close(got, ref, "rows, not causal")


@pytest.mark.parametrize("N,H,Hk,D", [(200, 8, 2, 256), (300, 96, 96, 128), (300, 96, 96, 64)])
@pytest.mark.parametrize("dtype", [C.F16, C.BF16])
def test_rows_climbing_scores(device, N, H, Hk, D, dtype):
    # scores that climb by > 11 log2 units per tile: rows re-base again and
    # again.  The other kernels' inputs, q scaled with sqrt(head_dim)
    c = C.prefill_case(1500 + D, N, H, Hk, D, 20, dtype)
    q, k = c["q"].copy(), c["k"].copy()
    q[:, :, 0] = 16.0 if D == 256 else 8.0
    k[:, :, 0] = 0.5 * np.arange(c["kv_len"], dtype=np.float32)[:, None]
    c["q"], c["qb"] = C.O.round_to(q, dtype)
    c["k"], c["kb"] = C.O.round_to(k, dtype)
    check(c, device, f"climbing scores, head_dim {D}")


# a later token's V that is not finite: the rows before it, whose weight for it is
# 0, do not take it in.  Token positions in the first and last tile of a wave, one
# past a tile, the last one (whose row fills up the tile), after a context and with
# split key ranges
@pytest.mark.parametrize("N,H,Hk,D,start,at", [
    (150, 16, 8, 256, 0, 5), (150, 16, 8, 256, 0, 149), (300, 8, 8, 256, 0, 33), (130, 32, 2, 256, 33, 65),
    (257, 6, 2, 200, 63, 95), (140, 4, 1, 256, 1000, 77), (33, 14, 2, 248, 900, 32), (5, 16, 8, 256, 1501, 2),
])
@pytest.mark.parametrize("dtype", [C.F16, C.BF16])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_wide_rows_hidden_v(device, N, H, Hk, D, start, at, dtype, bad):
    c = C.prefill_case(1900 + N + D, N, H, Hk, D, start, dtype)
    C.say(f"prefill rows, V not finite N={N} H={H} Hk={Hk} D={D} start={start} at={at} dtype={dtype} {bad}")
    q, k, v = (C.to_dev(c[x], dtype, device) for x in ("qb", "kb", "vb"))
    kvh, G = Hk - 1, H // Hk
    v[start + at, kvh] = bad
    out = mugen_amd.flash_prefill_attention(q, k, v, start, out_dtype=torch.float32).cpu().numpy()
    ref = C.prefill_ref(c, nthreads=16)  # of the finite V
    C.assert_close(out[:at], ref[:at], "rows before the token")
    if kvh:
        C.assert_close(out[:, :kvh * G], ref[:, :kvh * G], "the other kv heads")
    assert not np.isfinite(out[at:, kvh * G:]).any(), "rows that see it"


def exact(q, k, v):
    """Causal attention over a prompt in 64 bits, head by head."""
    N, H, D = q.shape
    G = H // k.shape[1]
    hidden = torch.ones(N, N, dtype=torch.bool, device=q.device).triu(1)
    out = torch.empty(N, H, D, dtype=torch.float64, device=q.device)
    for h in range(H):
        s = (q[:, h].double() @ k[:, h // G].double().T.contiguous()) / D ** 0.5
        out[:, h] = torch.softmax(s.masked_fill(hidden, float("-inf")), 1) @ v[:, h // G].double()
    return out


@pytest.mark.parametrize("N,H,Hk,D", [(150, 16, 8, 256), (300, 16, 8, 256), (300, 16, 4, 192)])
def test_rounding_of_the_weights(device, N, H, Hk, D):
    # f16 weights, f32 output.  Their rounding leaves 2^-11 / sqrt(3) x 0.72 (log-
    # uniform significands) = 2.0e-4 of the norm of sum p v, less what weights of
    # exactly 1 save: 1.35e-4 in prompts of a few hundred tokens with a reference
    # weight in each of four waves, 1.52e-4 with one.  The first tile's weights as
    # two terms: 1.1e-4
    g = torch.Generator(device=device).manual_seed(1700 + N)
    q, k, v = (torch.randn(s, generator=g, device=device).half() for s in ((N, H, D), (N, Hk, D), (N, Hk, D)))
    C.say(f"prefill rows, error against 64 bits N={N} D={D}")
    ref = exact(q, k, v)
    err = (mugen_amd.flash_prefill_attention(q, k, v, out_dtype=torch.float32).double() - ref).norm() / ref.norm()
    assert err.item() < 1.35e-4


def test_rounding_against_the_other_kernel(device):
    # 7 heads per kv head: the warp-specialised kernel's reference is the largest
    # of 64 scores, this kernel's of 32
    N, H, Hk, D = 2926, 28, 4, 128
    g = torch.Generator(device=device).manual_seed(1800)
    q, k, v = (torch.randn(s, generator=g, device=device).half() for s in ((N, H, D), (N, Hk, D), (N, Hk, D)))
    C.say("prefill rows and warp-specialised, error against 64 bits")
    ref = exact(q, k, v)
    err = [(mugen_amd.flash_prefill_attention(q, k, v, out_dtype=torch.float32, kernel=kernel).double() - ref).norm().item()
           for kernel in (0, _capi.PREFILL_KERNEL_WS)]
    assert err[0] <= err[1], err
