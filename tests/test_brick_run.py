"""CPU check of the runs into which the kernels split a brick's particles (csrc/brick_run.hpp), up to
the largest particle number."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("g++")


@pytest.mark.skipif(CXX is None, reason="no host C++ compiler")
def test_runs_cover_a_brick(tmp_path):
    exe = tmp_path / "brick_run_check"
    subprocess.run([CXX, "-O1", "-std=c++17", "-Wall", "-Werror", "-ftrapv", "-I",
                    os.path.join(ROOT, "latfield2_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp_host", "brick_run_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


def test_the_kernels_take_these_runs():
    """no kernel over a brick list forms the end of its run by itself"""
    csrc = os.path.join(ROOT, "latfield2_amd", "csrc")
    text = open(os.path.join(csrc, "bricks.hpp")).read() + open(os.path.join(csrc, "diffpm.hip")).read()
    assert "brick_run(" in text
    assert "r.p1" not in text
