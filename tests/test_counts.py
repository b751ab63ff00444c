"""The check of a history's outstanding flights at a push (tests/native/counts_check.cpp
over mt_counts.h, the header the cascade kernel includes): waves stop counting one by
one when the primaries are used up, and no valid run may be aborted for it."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_valid_pushes_pass_and_lost_counts_do_not(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = str(tmp_path / "counts_check")
    subprocess.run([hipcc, "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "mytrim_amd", "csrc"), "-o", exe,
                    os.path.join(HERE, "native", "counts_check.cpp")], check=True, capture_output=True)
    out = subprocess.run([exe, "20000"], check=True, capture_output=True, text=True).stdout
    r = {k: int(v) for k, v in (line.split() for line in out.strip().splitlines())}
    assert r["below"] > 0  # counts below 1 do occur in valid runs
    assert r["refused"] == 0
    assert r["corrupt"] == r["caught"] > 0  # and mean an error while primaries are left
