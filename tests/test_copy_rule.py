"""Which device-to-device copies the library's copy kernel takes: host only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_copies_the_kernel_takes_are_legal_launches():
    """tests/cpp/test_copy_rule.cpp compiles the rule (thrust_amd/csrc/copy_rule.hpp, which runtime.hip calls) for
    the host: no launch of 2^32 threads or more; larger copies, and ranges that reach beyond the allocation they
    begin in, are left to the runtime."""
    cpp = os.path.join(ROOT, "tests", "cpp")
    prog = os.path.join(cpp, "bin", "test_copy_rule")
    subprocess.run(["make", "-C", cpp, prog], check=True, capture_output=True)
    res = subprocess.run([prog], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0 and "PASSED" in res.stdout, res.stdout + res.stderr
