"""Bins of equal width of the merged selection (lvar_amd/csrc/score_bins.h): the arithmetic is shared by the kernel and by a
host program that lays the keys of a row out as the kernel does."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bins_are_ordered_and_hold_few_keys(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "score_bins_check")
    subprocess.run([cxx, "-O2", "-std=c++17", os.path.join(ROOT, "tests", "host", "score_bins_check.cpp"), "-o", exe],
                   check=True, timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.startswith("ok "), out.stdout + out.stderr
