"""4-bit store append, four lanes per group: row widths whose groups do not
fill a wave (and several waves' worth), and groups whose extremes tie across
the lanes' parts, byte for byte against the oracle's quantize_group."""
import numpy as np
import pytest
import torch

import mugen_amd
from oracle import oracle as O
from tests import cases as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hk,D", [(1, 32), (3, 32), (17, 32), (4, 128), (34, 32)])
def test_append_widths_and_ties(device, Hk, D):
    vpt, T = Hk * D, 40
    rng = np.random.default_rng(vpt)
    x = rng.standard_normal((2, T, vpt)).astype(np.float16)
    x[:, 1] = np.where(rng.random((2, vpt)) < 0.5, 0.0, -0.0)                    # only zeros of both signs
    x[:, 2] = np.where(rng.random((2, vpt)) < 0.5, 0.0, -0.0) + np.arange(vpt) % 32 // 31  # zeros tie for the min
    x[:, 3] = np.round(x[:, 3].astype(np.float32)).astype(np.float16)            # many ties
    x[:, 4] = 1.5                                                                # constant groups
    x[:, 5] = rng.standard_normal((2, vpt)).astype(np.float16) * np.float16(6e-8)  # subnormals
    x[:, 6, ::32] = 60000.0
    bits = x.view(np.uint16)
    kv = mugen_amd.KVCacheQ4(1, 2, Hk, D, max_seq_len=64, fp16_preserve_last=4, max_new=8, device=device)
    C.say(f"kv_q4 append vpt={vpt}")
    dev = lambda b: torch.from_numpy(np.ascontiguousarray(b).view(np.float16)).to(device)
    for t in range(0, T, 8):
        kv.append(0, dev(bits[:, t:t + 8]), dev(bits[::-1, t:t + 8]))
        kv.advance()
    torch.cuda.synchronize()
    for b in range(2):
        for got, src in ((kv.q4_k, bits[b]), (kv.q4_v, bits[1 - b])):
            want = O.q4_quantize_tokens(src[:T - 4])
            assert np.array_equal(got[0][b, :T - 4].cpu().numpy(), want), f"vpt {vpt} seq {b}"
