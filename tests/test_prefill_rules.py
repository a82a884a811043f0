"""Which prefill kernel takes a prompt (mugen_amd/csrc/prefill_rules.h), compiled
for the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("rules") / "prefill_rules_check")
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", os.path.join(ROOT, "mugen_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "prefill_rules_check.cpp"), "-o", exe], check=True)

    def run(*shape, args=()):
        return subprocess.run([exe, *args], input=" ".join(map(str, shape)) + "\n", check=True, capture_output=True,
                              text=True).stdout.strip()
    return run


@pytest.mark.parametrize("N,H,Hk,D,kernel", [
    (256, 32, 8, 64, "block"), (1023, 8, 2, 64, "block"), (1024, 8, 2, 64, "ws"), (4096, 8, 2, 64, "ws"),
    # few kv heads: long prompts that make too few flattened-row blocks
    (4097, 8, 2, 64, "block"), (9900, 8, 2, 64, "block"), (9000, 9, 3, 64, "block"), (20000, 4, 1, 64, "block"),
    (16000, 2, 1, 64, "block"),
    (64, 14, 2, 64, "ws"), (5000, 14, 2, 64, "ws"), (16, 28, 4, 128, "ws"), (2900, 28, 4, 128, "ws"), (700, 8, 2, 96, "ws"),
    # from 128-row blocks enough on, the flattened-row kernel
    (2926, 28, 4, 128, "rows"), (2048, 32, 8, 128, "rows"), (2047, 8, 8, 128, "ws"), (4096, 8, 8, 128, "rows"),
    (1024, 32, 16, 128, "rows"), (2560, 32, 8, 64, "rows"), (5860, 14, 2, 64, "rows"), (1024, 32, 32, 64, "rows"),
    # two heads per kv head at head_dim 64; full slots of one kv head
    (2048, 16, 8, 64, "ws"), (2560, 16, 8, 64, "rows"), (8192, 4, 2, 64, "block"), (12288, 4, 2, 64, "rows"),
    (24576, 2, 1, 64, "block"), (28672, 2, 1, 64, "rows"), (20500, 4, 1, 64, "block"), (26000, 4, 1, 64, "rows"),
    (10300, 8, 1, 64, "ws"), (12800, 8, 1, 64, "rows"),
    # 8 heads per kv head, full slots
    (5180, 16, 2, 128, "ws"), (6144, 16, 2, 128, "rows"), (2620, 32, 4, 128, "rows"),
    # above head_dim 128: a workgroup per (token, kv head) pair, one round of them at
    # 256, two at the padded widths, one with many heads
    (32, 16, 8, 256, "pairs"), (33, 16, 8, 256, "rows"), (1021, 16, 8, 256, "rows"), (256, 1, 1, 256, "pairs"),
    (257, 1, 1, 256, "rows"), (300, 1, 1, 136, "pairs"), (513, 1, 1, 136, "rows"), (64, 16, 8, 192, "pairs"),
    (65, 16, 8, 192, "rows"), (128, 16, 4, 192, "pairs"), (129, 16, 4, 192, "rows"), (17, 128, 16, 136, "rows"),
    (33, 64, 8, 192, "rows"), (17, 64, 16, 192, "rows"),
])
def test_prompt_kernel(choose, N, H, Hk, D, kernel):
    assert choose(N, 0, 1, H, Hk, D) == kernel


# blocks of about the same key count: after a long context, or not causal
@pytest.mark.parametrize("N,H,Hk,D,kernel", [
    (2933, 28, 4, 128, "ws"), (3518, 28, 4, 128, "rows"), (2568, 32, 4, 128, "ws"), (3072, 32, 4, 128, "ws"), (4400, 32, 4, 128, "rows"),
    (2048, 16, 8, 64, "rows"), (16384, 2, 1, 64, "block"), (20500, 4, 1, 64, "rows"), (3421, 24, 4, 128, "rows"), (2926, 28, 4, 64, "rows"),
    (17, 64, 16, 192, "pairs"), (33, 64, 8, 192, "rows"), (33, 16, 8, 256, "rows"),
])
def test_level_chunk_kernel(choose, N, H, Hk, D, kernel):
    assert choose(N, N, 1, H, Hk, D) == kernel and choose(N, 0, 0, H, Hk, D) == kernel


def test_row_numbers_fit_32_bits(choose):
    # 2^31 rows of a kv head: the kernel's row numbers would overflow
    assert choose(2**27 - 8, 0, 0, 16, 1, 8) == "rows" and choose(2**27, 0, 0, 16, 1, 8) == "ws"


@pytest.mark.parametrize("slots", [1, 7, 8, 31, 33, 255, 3 * 17 * 5, 100 * 16 * 8])
@pytest.mark.parametrize("part", [2 * 8, 2 * 128, 4 * 136, 4 * 256])
def test_split_partials_are_aligned(choose, slots, part):
    # one token, one head, 7 key ranges: the pairs end 56 bytes past the boundary
    at, size = map(int, choose(slots, part, args=("partials",)).split())
    assert at % 16 == 0 and at >= 8 * slots
    assert 255 + at + slots * part <= size, "the workspace covers both roundings"
