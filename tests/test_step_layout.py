"""Who does what in a decode step in one launch (csrc/step_layout.h), checked with g++ from tests/step_layout_check.cpp: no GPU
needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_step_layout(tmp_path):
    exe = tmp_path / "step_layout_check"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", os.path.join(ROOT, "tests", "step_layout_check.cpp"), "-o", str(exe)])
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "step layout ok" in r.stdout, r.stdout + r.stderr
