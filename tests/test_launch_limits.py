"""Launches over many rows are folded so that no grid passes 2^32 - 1 threads in
a dimension, which HIP refuses (tests/cpp/launch_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_rows_per_launch(tmp_path):
    exe = str(tmp_path / "launch_check")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(HERE, "cpp", "launch_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and "launch check ok" in r.stdout, r.stdout
