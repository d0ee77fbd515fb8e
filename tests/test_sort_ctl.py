"""The control block of a radix sort, on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_nothing_runs_behind_a_pass_that_gave_up():
    """tests/cpp/test_sort_ctl.cpp compiles the control block (thrust_amd/csrc/sort_ctl.hpp, whose functions the
    kernels call) for the host: whichever pass stops waiting, no later launch touches the array."""
    cpp = os.path.join(ROOT, "tests", "cpp")
    prog = os.path.join(cpp, "bin", "test_sort_ctl")
    subprocess.run(["make", "-C", cpp, prog], check=True, capture_output=True)
    res = subprocess.run([prog], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and "PASSED" in res.stdout, res.stdout + res.stderr
