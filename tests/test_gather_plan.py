"""The host arithmetic of the gather launches (gelib_amd/csrc/gather_plan.h) at extents of tens of gigabytes, which a test
cannot allocate: a small C++ program prints what would be launched."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "gather_plan_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "gelib_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", "gather_plan_check.cpp"), "-o", exe])
    return lambda *args: subprocess.check_output([exe] + [str(a) for a in args], text=True).split("\n")[0]


@pytest.mark.parametrize("n,aligned,vec", [(1 << 16, 1, 2), ((1 << 16) + 2, 1, 2), (80000, 1, 2), (1 << 15, 0, 1), (46341, 1, 1)])
def test_last_thread_owns_the_end_of_a_large_slice(check, n, aligned, vec):
    """One target whose slice is n x n complex numbers (9 to 51 GB): the last thread's elements are the slice's last."""
    want = n * n
    assert check("cover", 1, 1, n, 1, n, 1, aligned) == "%d %d %d" % (vec, want // vec, want - vec)
