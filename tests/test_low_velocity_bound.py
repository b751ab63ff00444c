"""The energy below which the heavy-ion stopping takes its low-velocity branch for
sure (StopConst::e_low) against a bisection of the reference's expressions."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
BUILD = os.path.join(ROOT, "mytrim_amd", "_build")


def test_bound_below_and_close_to_the_branch(tmp_path):
    gxx = shutil.which("g++")
    if not gxx or not os.path.exists(os.path.join(BUILD, "mt_scoef_default.inc")):
        pytest.skip("g++ or the built tables not available")
    exe = str(tmp_path / "elow_check")
    csrc = os.path.join(ROOT, "mytrim_amd", "csrc")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I" + csrc, "-I" + os.path.join(ROOT, "include"), "-I" + BUILD, "-o",
                    exe, os.path.join(HERE, "native", "elow_check.cpp"), os.path.join(csrc, "mt_host.cpp")],
                   check=True, capture_output=True)
    rows = [line.split() for line in subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()]
    assert len(rows) == 90 * 8
    some = 0
    for row in rows:
        z1, z2, bound, exact, vf = (float(x) for x in row)
        # never above the branch's own limit, and below it by the margin of 1e-5
        # of vr alone: above the Fermi velocity 3e-5 of e; below it, where vr is
        # flat, 1e-5 vr / (d vr / de) <= 7.5e-4 vf^2; 1e-6 and the float's
        # rounding come on top
        assert bound <= exact, (z1, z2)
        if exact > 0.0:
            some += 1
            assert bound >= exact * (1.0 - 4e-5) - 8e-4 * vf * vf, (z1, z2, bound, exact)
    assert some > 500
