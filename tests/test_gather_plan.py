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


@pytest.mark.parametrize("n,aligned,threads", [
    ((1 << 32) - 256, 0, (1 << 32) - 256),      # 8 bytes a thread: the largest whole number of blocks
    ((1 << 32) - 255, 0, None),                 # one thread more is a block more
    ((1 << 32) - 1, 0, None),
    ((1 << 33) - 512, 1, (1 << 32) - 256),      # 16 bytes a thread
    ((1 << 33) - 510, 1, None),
])
def test_a_part_fits_a_launch_or_is_left_to_the_other_kernel(check, n, aligned, threads):
    """A launch holds fewer than 2^32 threads, in whole blocks of 256; one target of n complex numbers."""
    got = check("cover", 1, 1, 1, 1, n, 0, aligned)
    assert got.split()[-2:-1] == ([] if threads is None else [str(threads)]), got


@pytest.mark.parametrize("threads", [[1 << 31] * 2, [1 << 31] * 5, [(1 << 32) - 256] * 3, [100] * 19, [(1 << 32) - 512, 256, 256],
                                     [1 << 30, 3 << 29, 1, 1 << 31, 257]])
def test_no_launch_holds_more_threads_than_a_launch_may(check, threads):
    launches = [tuple(map(int, item.split(":"))) for item in check("pack", *threads).split()]
    assert sum(p for p, _ in launches) == len(threads)
    assert sum(b for _, b in launches) == sum((t + 255) // 256 for t in threads)
    for parts, blocks in launches:
        assert 1 <= parts <= 8 and blocks * 256 < 1 << 32
