"""Binned mode's bins (axiomr_amd/csrc/bins.hpp, the functions that the
kernels call) on the CPU: the levels of a bin's entries at every first-level
size, the permutation of the bins' counters, and waves whose entries lie in
levels that other waves open, the slots handed out in any order: every wait
ends and every entry is in its place."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "native" / "test_bins.cpp"


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_bin_layout(tmp_path):
    exe = tmp_path / "bins"
    cmd = ["g++", "-std=c++17", "-O1", "-g", "-Wall", "-Wno-unknown-pragmas", "-pthread", "-o", str(exe), str(SRC)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and not r.stderr, r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout + r.stderr
