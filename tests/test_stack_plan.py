"""The stacked passes' tables on the CPU: interpreted window by window (every
access bounds-checked) against single merges, bit for bit, at every depth and
first iteration of odd, even, stepped and legacy plans (tests/cpp/stack_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_stack_tables_against_single_merges(tmp_path):
    exe = tmp_path / "stack_check"
    src = [os.path.join(ROOT, "tests", "cpp", "stack_check.cpp"),
           os.path.join(ROOT, "cpp_projects_amd", "csrc", "stack_plan.cpp"),
           os.path.join(ROOT, "cpp_projects_amd", "csrc", "plan.cpp")]
    r = subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-ffp-contract=off", "-fsanitize=address,undefined",
                        "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "include"), *src, "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0 and "stack check ok" in r.stdout, (r.stdout + r.stderr)[-3000:]
