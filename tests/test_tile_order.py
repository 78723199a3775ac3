"""Order of the query tiles of a plain attention launch (lvar_amd/csrc/tile_order.h): the integer arithmetic is shared by
the kernel and by a host program that walks every workgroup of a launch."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_tile_once_and_no_xcd_over_its_share(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "tile_order_check")
    subprocess.run([cxx, "-O2", "-std=c++17", os.path.join(ROOT, "tests", "host", "tile_order_check.cpp"), "-o", exe],
                   check=True, timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.startswith("ok "), out.stdout + out.stderr


def test_form_of_a_launch_on_both_sides_of_every_bound(tmp_path):
    """lvar_amd/csrc/launch_forms.h: the rules that the launch code takes its form of workgroup from."""
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "launch_forms_check")
    subprocess.run([cxx, "-O2", "-std=c++17", os.path.join(ROOT, "tests", "host", "launch_forms_check.cpp"), "-o", exe],
                   check=True, timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and out.stdout.startswith("ok "), out.stdout + out.stderr
