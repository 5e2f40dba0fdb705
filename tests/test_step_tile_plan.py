"""The planner of the fused per-step kernel's tiles (gpuvoxels_amd/csrc/vx3h_steptile.cpp),
on the CPU: every voxel owned once, tiles within a workgroup's threads and slots, surface
voxels first, neighbour slots and halo at the right voxels, every link kept by the tile of
its negative end and listed, with that state, by the tile of its positive end
(tests/step_tile_check.cpp)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from gpuvoxels_amd import engine, workloads
from test_tile_plan import lattice

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "gpuvoxels_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    exe = str(tmp_path_factory.mktemp("steptile") / "step_tile_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe, os.path.join(HERE, "step_tile_check.cpp"),
                    os.path.join(CSRC, "vx3h_steptile.cpp")], check=True)
    return exe


def plan(program, m):
    vneg, vpos, axis, _ = engine.topology(m)
    lines = ["%d %d" % (len(m.ijk), len(vneg))]
    lines += ["%d %d %d" % tuple(r) for r in m.ijk]
    lines += ["%d %d %d" % (a, b, c) for a, b, c in zip(vneg, vpos, axis)]
    r = subprocess.run([program], input="\n".join(lines) + "\n", stdout=subprocess.PIPE, text=True, check=True, timeout=120)
    out = r.stdout.split()
    assert out[0] == "ok", out
    return [int(x) for x in out[1:]]


def box(nx, ny, nz):
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    return lattice(np.stack([x.ravel(), y.ravel(), z.ravel()], 1))


@pytest.mark.parametrize("shape", [(1, 1, 1), (256, 1, 1), (257, 1, 1), (8, 8, 5), (7, 9, 11), (32, 32, 6), (61, 47, 3)])
def test_boxes(program, shape):
    tiles, halo, incoming = plan(program, box(*shape))
    assert (tiles == 1) == (np.prod(shape) <= 256)
    if shape == (32, 32, 6):   # 8 x 8 x 3 blocks
        assert tiles == 32


@pytest.mark.parametrize("radius,count", [(1, 40), (2, 40), (3, 9), (4, 6), (5, 3)])
def test_separate_bodies_stay_whole(program, radius, count):
    m = workloads.arena_balls(count, radius=radius, arena=90, steps=0, seed=1)
    tiles, halo, incoming = plan(program, m)
    n = len(workloads.ball_offsets(radius))
    if n <= 288:   # two of more than 32 voxels do not share a tile, here
        assert halo == 0 and incoming == 0
        assert tiles == count if n > 32 else tiles < count


@pytest.mark.parametrize("grid,seed", [(5, 1), (12, 2), (23, 3)])
def test_robots(program, grid, seed):
    plan(program, workloads.robot(np.random.default_rng(seed), grid=grid, steps=0))
