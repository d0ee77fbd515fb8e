"""The searches for a merge's tile boundaries, on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_boundaries_in_order_and_tiles_inside_the_ranges():
    """tests/cpp/test_merge_search.cpp compiles include/thrust/system/hip/detail/merge_search.h, whose steps the kernels
    take, for the host: every group size finds the boundaries of sorted keys, and in keys that are in no order (NaN among
    them) no tile reads outside the two ranges."""
    cpp = os.path.join(ROOT, "tests", "cpp")
    prog = os.path.join(cpp, "bin", "test_merge_search")
    subprocess.run(["make", "-C", cpp, prog], check=True, capture_output=True)
    res = subprocess.run([prog], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and "PASSED" in res.stdout, res.stdout + res.stderr
