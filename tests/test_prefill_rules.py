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

    def run(*shape):
        return subprocess.run([exe], input=" ".join(map(str, shape)) + "\n", check=True, capture_output=True,
                              text=True).stdout.strip()
    return run


@pytest.mark.parametrize("N,H,Hk,D,kernel", [
    (256, 32, 8, 64, "block"), (1023, 8, 2, 64, "block"), (1024, 8, 2, 64, "ws"), (4096, 8, 2, 64, "ws"),
    # few kv heads: long prompts that make too few flattened-row blocks
    (4097, 8, 2, 64, "block"), (9900, 8, 2, 64, "block"), (9000, 9, 3, 64, "block"), (20000, 4, 1, 64, "block"),
    (16000, 2, 1, 64, "block"),
    (64, 14, 2, 64, "ws"), (5000, 14, 2, 64, "ws"), (16, 28, 4, 128, "ws"), (2900, 28, 4, 128, "ws"), (700, 8, 2, 96, "ws"),
])
def test_prompt_kernel(choose, N, H, Hk, D, kernel):
    assert choose(N, H, Hk, D) == kernel
