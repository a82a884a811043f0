"""The context-split plan that decode calls without host lengths make on the
device: its arithmetic, compiled for the host (tests/cpp/split_plan_check.cpp),
never gives a work list that the launch's workgroups do not cover."""
import os
import shutil
import subprocess

import pytest

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
