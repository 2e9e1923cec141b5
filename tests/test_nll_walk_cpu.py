"""The nll_loss gradient over short rows (csrc/rocm/nll_walk.h) on the CPU: no
read of a target or a weight past its array, whatever the last target is.
Compiled from tests/native/nll_walk_test.cpp with g++ and run."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.path.join(os.path.dirname(HERE), "tensorplay_amd", "csrc", "rocm")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_reads_stay_in_range(tmp_path):
    exe = str(tmp_path / "nll_walk_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", ROCM,
                    os.path.join(HERE, "native", "nll_walk_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    print(r.stdout, r.stderr)
    assert r.returncode == 0 and "OK" in r.stdout
