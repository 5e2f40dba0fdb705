"""Plans of the fused per-step kernel's tiles beside other simulations, on the CPU: the same
invariants (tests/step_tile_check.cpp) with fuller tiles, and the line past which bodies too
small and too far apart to share tiles stay on the per-step kernels."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from gpuvoxels_amd import workloads
from test_step_tile_plan import CSRC, HERE, plan, program  # noqa: F401
from test_tile_plan import lattice


@pytest.fixture(scope="module")
def beside(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("steptile") / "step_tile_beside_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "step_tile_beside_check.cpp"),
                    os.path.join(CSRC, "vx3h_steptile.cpp")], check=True)
    return exe


@pytest.mark.parametrize("count,radius,arena", [(100, 2, 50), (40, 1, 30), (30, 3, 40), (9, 4, 30)])
def test_fuller_tiles(program, beside, count, radius, arena):  # noqa: F811
    m = workloads.arena_balls(count, radius=radius, arena=arena, steps=0, seed=2)
    alone, among = plan(program, m)[0], plan(beside, m)[0]
    assert among < alone if radius < 3 else among <= alone


def test_one_body_is_cut_alike(program, beside):  # noqa: F811
    z, y, x = np.meshgrid(np.arange(9), np.arange(14), np.arange(11), indexing="ij")
    m = lattice(np.stack([x.ravel(), y.ravel(), z.ravel()], 1))
    assert plan(program, m) == plan(beside, m)


def test_when_tiles_pay(tmp_path):
    """Both sides of the line: what was measured faster on the fused kernel, and what was not."""
    src = tmp_path / "pay.cpp"
    src.write_text('#include <cstdio>\n#include "%s"\nint main() {\n    long long t, v;\n    size_t r;\n'
                   '    while (scanf("%%lld %%lld %%zu", &t, &v, &r) == 3) printf("%%d", (int)vx3::stepTilesPay(t, v, r));\n}\n'
                   % os.path.join(CSRC, "vx3h_steptile.h"))
    exe = str(tmp_path / "pay")
    subprocess.run(["g++", "-std=c++17", "-o", exe, str(src)], check=True)
    faster = [(979, 2000, 8), (979, 2000, 4), (865, 16000, 4), (1876, 108000, 4), (1876, 108000, 8), (3980, 264000, 8),
              (4494, 512000, 4), (2048, 2048 * 257, 8), (10923, 128 ** 3, 4), (1, 1, 8)]
    slower = [(2000, 4000, 8), (2000, 4000, 4), (4000, 8000, 8), (1740, 32000, 8), (1740, 32000, 4), (3980, 264000, 4),
              (2 ** 22, 2 ** 23, 8)]
    lines = "\n".join("%d %d %d" % c for c in faster + slower)
    out = subprocess.run([exe], input=lines, stdout=subprocess.PIPE, text=True, check=True).stdout
    assert out == "1" * len(faster) + "0" * len(slower)


def test_when_rebuilds_pay(tmp_path):
    src = tmp_path / "pay.cpp"
    src.write_text('#include <cstdio>\n#include "%s"\nint main() {\n    long long t, s;\n'
                   '    while (scanf("%%lld %%lld", &t, &s) == 2) printf("%%d", (int)vx3::stepRebuildsPay(t, s));\n}\n'
                   % os.path.join(CSRC, "vx3h_steptile.h"))
    exe = str(tmp_path / "pay")
    subprocess.run(["g++", "-std=c++17", "-o", exe, str(src)], check=True)
    out = subprocess.run([exe], input="1 1\n65536 65536\n36864 6500\n131072 131072\n4194303 4194303\n4194303 100\n",
                         stdout=subprocess.PIPE, text=True, check=True).stdout
    assert out == "111001"
