"""The context-split plan that decode calls without host lengths make on the
device: its arithmetic, compiled for the host (tests/cpp/split_plan_check.cpp),
never gives a work list that the launch's workgroups do not cover.  And the plan
of the 4-bit store with host lengths, by its workspace size."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from mugen_amd import _capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("plan") / "split_plan_check")
    subprocess.run([cxx, "-std=c++17", "-O2", "-I", os.path.join(ROOT, "mugen_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "split_plan_check.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
def test_work_list_fits(check, seed):
    r = subprocess.run([check, str(seed), "100000"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout


def store_splits(lens, H, Hk, D=128, cache=8192):
    a = _capi.GqaDecodeQ4Args()
    a.q = a.seq_lens = a.n_q4 = a.out = 0x1000
    a.store.q4_k = a.store.q4_v = a.store.ring_k = a.store.ring_v = 0x1000
    a.store.q4_seq_stride, a.store.ring_seq_stride = cache * Hk * D // 32 * 20, 512 * Hk * D
    a.store.ring, a.store.fp16_preserve_last = 512, 256
    a.batch, a.n_heads, a.n_kv_heads, a.head_dim, a.max_seq_len, a.out_dtype = len(lens), H, Hk, D, cache, _capi.F16
    lens = np.asarray(lens, np.int32)
    a.seq_lens_host = lens.ctypes.data
    size = _capi.lib().mugen_attn_gqa_decode_q4_workspace_size(ctypes.byref(a))
    return (size - 256) // (len(lens) * H * (4 * D + 8))


# 1024-token items: the longest sequence in 8, one more for the f16 tokens
@pytest.mark.parametrize("B,H,Hk,lo,hi,deep", [
    (64, 28, 4, 512, 8191, True), (24, 32, 8, 512, 8191, True), (32, 32, 8, 8191, 8191, True),
    (32, 28, 4, 512, 8191, True),
    # the round's own chunk is short: the store's extra split per sequence costs
    # more than the even load gains
    (12, 32, 8, 3000, 8191, False), (24, 28, 4, 512, 8191, False), (48, 8, 2, 3000, 8191, False),
    (16, 32, 8, 512, 8191, False),
])
def test_store_plan_of_large_batches(B, H, Hk, lo, hi, deep):
    lens = np.random.default_rng(B).integers(lo, hi + 1, B)
    splits = store_splits(lens, H, Hk)
    assert (splits == -(-int(lens.max()) // 1024) + 1) == deep, splits
