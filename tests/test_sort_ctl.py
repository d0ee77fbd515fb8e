"""The control block of a radix sort and the rule of its two-digit way, on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(name):
    cpp = os.path.join(ROOT, "tests", "cpp")
    prog = os.path.join(cpp, "bin", name)
    subprocess.run(["make", "-C", cpp, prog], check=True, capture_output=True)
    res = subprocess.run([prog], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and "PASSED" in res.stdout, res.stdout + res.stderr


def test_nothing_runs_behind_a_pass_that_gave_up():
    """tests/cpp/test_sort_ctl.cpp compiles the control block (thrust_amd/csrc/sort_ctl.hpp, whose functions the
    kernels call) for the host: whichever pass stops waiting, no later launch touches the array."""
    _run("test_sort_ctl")


def test_kinds_of_keys_that_take_the_two_digit_way():
    """tests/cpp/test_top_digits.cpp compiles the rule (thrust_amd/csrc/top_digits.hpp, which the plan kernel
    calls) for the host: random keys take the way, keys whose stretches do not fit do not."""
    _run("test_top_digits")
