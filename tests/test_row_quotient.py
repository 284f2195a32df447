"""The quotient of the int8 family's decode rule (csrc/row_quotient.h) is the IEEE one: checked with g++ from tests/row_quotient_check.cpp, no GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_row_quotient(tmp_path):
    exe = tmp_path / "row_quotient_check"
    fma = ["-mfma"] if "fma" in open("/proc/cpuinfo").read().split() else []
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-Wno-unknown-pragmas", "-ffp-contract=off", *fma, "-pthread",
                           os.path.join(ROOT, "tests", "row_quotient_check.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "row quotient ok" in r.stdout, r.stdout + r.stderr
