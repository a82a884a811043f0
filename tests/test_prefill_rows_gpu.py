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


def test_wide_rows_not_causal(device):
    c = C.prefill_case(1400, 140, 8, 4, 256, 53, C.F16)
    got, _ = run(c, device, causal=False)
    N, H, Hk, D, kv = 140, 8, 4, 256, c["kv_len"]
    ref = C.O.gqa_attention(c["q"], c["k"].reshape(1, kv, Hk, D).repeat(N, 0), c["v"].reshape(1, kv, Hk, D).repeat(N, 0),
                            [kv] * N, H, Hk, D, kv * Hk * D)
    C.assert_close(got, ref, "rows, not causal")


@pytest.mark.parametrize("dtype", [C.F16, C.BF16])
def test_wide_rows_climbing_scores(device, dtype):
    # scores that climb by > 15 log2 units per tile: the re-base runs on every
    # tile.  The same inputs as the other kernels' test, scaled for head_dim 256
    c = C.prefill_case(1500, 200, 8, 2, 256, 20, dtype)
    q, k = c["q"].copy(), c["k"].copy()
    q[:, :, 0] = 16.0
    k[:, :, 0] = 0.5 * np.arange(c["kv_len"], dtype=np.float32)[:, None]
    c["q"], c["qb"] = C.O.round_to(q, dtype)
    c["k"], c["kb"] = C.O.round_to(k, dtype)
    check(c, device, "climbing scores, head_dim 256")
