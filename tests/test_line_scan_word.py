"""Host test of the large-N scans' word extraction (line_scan_word_test.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "accrqa_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_line_scan_word(tmp_path):
    exe = tmp_path / "line_scan_word_test"
    subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-I", CSRC, os.path.join(HERE, "line_scan_word_test.cpp"), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.strip().endswith("ok")
