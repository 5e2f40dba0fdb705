"""The one-workgroup kernel with the links of all axes at once against the per-step kernels,
which vx3h_batch_step_noalloc runs on every simulation: the same operations in the same order,
so the same bits.  Sizes at the edges of its shapes (768 voxels and 768 or 960 links in FP64,
1,024 voxels and 1,024 or 1,984 links in FP32) and one past them, where the kernel that goes
axis by axis takes over; no link at all; more simulations than compute units; short launches."""
import numpy as np
import pytest

from gpuvoxels_amd import _abi, engine, workloads
from gpuvoxels_amd.model import Ext

pytestmark = pytest.mark.gpu

KEYS = ("pos", "orient", "lin_mom", "ang_mom", "flags", "tfac", "strain", "max_strain", "small_angle")


def body(plate, bar):
    """A plate of plate[0] x plate[1] voxels and a bar of `bar` beside it; several phases, an
    external on each, a fixed and a failing material."""
    a, n = plate
    m = workloads.slab(3, 3, 1, steps=0, collisions=False)
    xy = [(x, y, 0) for y in range(n) for x in range(a)] + [(x, n + 3, 0) for x in range(bar)]
    m.ijk = np.array(xy, np.int32)
    m.mat = np.zeros(len(xy), np.int32)
    m.phase = np.round(np.linspace(0, 1, len(xy)) * 30) / 30
    ext = [Ext(voxel=0, dof_fixed=63, translate=(0.0, 0.0, 0.001), rotate=(0.0, 0.1, 0.0))]
    if len(xy) > 1:
        ext.append(Ext(voxel=len(xy) - 1, dof_fixed=5, force=(0.0, 0.02, 0.0)))
    m.externals = ext
    return m


def sizes(m):
    return m.n_voxels, len(engine.topology(m)[0])


def robots(n, grid):
    rng = np.random.default_rng(5)
    out = []
    for i in range(n):
        m = workloads.robot(rng, grid=grid, steps=0)
        m.materials[1].fixed = i % 2
        m.materials[2].mat_model, m.materials[2].fail_stress = _abi.MDL_LINEAR_FAIL, 800.0
        out.append(m)
    return out


def check(models, precision, chunks):
    got = []
    for noalloc in (False, True):
        b = engine.Batch(precision=precision, path=_abi.PATH_AUTO)
        slots = [b.admit(m) for m in models]
        assert all(b.workgroups(s) == 1 for s in slots) or len(models) == 1   # (an edge's far side may be tiled)
        for n in chunks:
            (b.step_noalloc if noalloc else b.step)(n)
        st = b.poll()
        got.append([(b.read_state(s, nl=max(sizes(m)[1], 1)), st[s]) for m, s in zip(models, slots)])
        b.close()
    for (x, sx), (y, sy) in zip(*got):
        assert sx.steps == sy.steps and sx.state == sy.state and sx.current_time == sy.current_time
        for k in KEYS:
            assert np.array_equal(x[k], y[k], equal_nan=True), k


F64, F32 = _abi.PREC_F64, _abi.PREC_F32


@pytest.mark.parametrize("precision,plate,bar,expect", [
    (F64, (1, 1), 0, (1, 0)), (F64, (20, 18), 87, (447, 768)), (F64, (20, 18), 88, (448, 769)), (F64, (20, 18), 279, (639, 960)),
    (F64, (20, 18), 280, (640, 961)), (F64, (3, 3), 759, (768, 770)), (F64, (3, 3), 760, (769, 771)),
    (F32, (20, 25), 70, (570, 1024)), (F32, (20, 25), 71, (571, 1025)), (F32, (31, 33), 0, (1023, 1982)), (F32, (31, 33), 1, (1024, 1982)),
    (F32, (31, 33), 2, (1025, 1983))])
def test_edges(precision, plate, bar, expect):
    m = body(plate, bar)
    assert sizes(m) == expect
    check([m], precision, [1, 2, 60])


@pytest.mark.parametrize("precision", [F64, F32])
def test_several(precision):
    cube = workloads.cube(6, steps=0)
    line = body((1, 1), 40)
    check(robots(4, 7) + [cube, line] + robots(2, 10), precision, [150, 33])


@pytest.mark.parametrize("precision,grid", [(F64, 4), (F32, 12)])
def test_more_than_compute_units(precision, grid):
    check(robots(300, grid), precision, [40, 5])
