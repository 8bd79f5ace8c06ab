"""Sizes of the march's buffers (eik_march_size.h), by mode: the instances' lists do not overlap and end
within their buffer, and small grids take what their lists need (a workgroup per source once took
2.3 MB of list for 61x44 nodes, and a no-allocation call then marched 55 sources at most).  Host build."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "eikonalsolvers.jl_amd", "csrc")


def test_march_lists_fit_and_small_grids_stay_small(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path / "march_size_test")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", CSRC, "-o", exe, os.path.join(HERE, "host", "march_size_test.cpp")],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
