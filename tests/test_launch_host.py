"""Launch extents of the fills (eik_launch.h): a launch's blocks x threads is a 32-bit number, and the
pending buffers of one call exceed it (3 x 1.43e9 nodes: 331 sources on 201x201x101).  Host build of
the rule."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "eikonalsolvers.jl_amd", "csrc")


def test_fill_extents_stay_within_32_bits(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path / "launch_test")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", CSRC, "-o", exe, os.path.join(HERE, "host", "launch_test.cpp")],
                   check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_no_fill_is_launched_by_element_count():
    """Every fill goes through the one helper that bounds its grid."""
    for f in sorted(os.listdir(CSRC)):
        with open(os.path.join(CSRC, f)) as h:
            s = h.read()
        n = s.count("k_fill") - s.count("k_fill(") if f != "eik_internal.h" else 0
        assert n == 0, f"{f} launches a fill kernel itself"
