"""The contact loops' early test as the kernels compile it (gpuvoxels_amd/csrc/vx3_pair.h)
leaves out only pairs whose contact force is zero (tests/pair_check.cpp, on the CPU)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_only_zero_forces(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path / "pair_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-Wall", "-o", exe, os.path.join(HERE, "pair_check.cpp")], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, check=True, timeout=120).stdout.split()
    assert out[0] == "ok", out
    assert int(out[1]) > 20000
