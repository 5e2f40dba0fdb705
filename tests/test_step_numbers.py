"""The numbers of the fused kernel's step reports past the largest 32-bit one, which a long-lived
batch reaches (tests/step_number_check.cpp, on the CPU)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_numbers_start_over(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path / "step_number_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", exe, os.path.join(HERE, "step_number_check.cpp")], check=True)
    out = subprocess.run([exe], stdout=subprocess.PIPE, text=True, check=True, timeout=60).stdout.split()
    assert out[0] == "ok", out
    assert int(out[1]) >= 59
