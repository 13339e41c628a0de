"""Host unit test of the run extraction the kernels compile, consume_word() of
accrqa_amd/csrc/rqa_bits.hpp, against a direct scan, and of the skip of
threshold pairs (line_scan_run_test.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "accrqa_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_line_scan_run(tmp_path):
    exe = str(tmp_path / "line_scan_run_test")
    subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-I", CSRC, os.path.join(HERE, "line_scan_run_test.cpp"), "-o", exe],
                   check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.strip().endswith("ok")
