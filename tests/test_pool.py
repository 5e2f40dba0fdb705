"""The ranges of the device pools when an array cannot be enlarged: nothing is taken, in one
pool or in several at once, so nothing later is placed past an array's end or released twice
(tests/pool_check.cpp, on the CPU)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_ranges_survive_failed_growth(tmp_path, seed):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path / "pool_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-o", exe,
                    os.path.join(HERE, "pool_check.cpp")], check=True)
    out = subprocess.run([exe, str(seed)], stdout=subprocess.PIPE, text=True, check=True, timeout=60).stdout.split()
    assert out[0] == "ok", out
    assert int(out[1]) > 50
