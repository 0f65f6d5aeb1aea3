"""Launches that split their sources take fewer splits where memory does not
hold the workspace of all (flowvpm.jl_amd/csrc/uj_split.h): the search against
amounts of memory from what every split takes down to less than one takes, on
the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_fewer_splits(tmp_path):
    exe = str(tmp_path / "split_driver")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I" + os.path.join(ROOT, "flowvpm.jl_amd", "csrc"),
                    os.path.join(ROOT, "tests", "sanitize", "split_driver.cpp"), "-o", exe],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "split_driver OK" in r.stdout, r.stdout + r.stderr
