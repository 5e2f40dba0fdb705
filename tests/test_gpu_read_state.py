"""Reading simulations' state back: pieces of 256 voxels or links, several launches for a
large simulation, several simulations in a batch.  Known values before the first step;
afterwards the same simulation alone, at other places of the device arrays, in the other
order; positions against the sums that the status reports (exact: the same additions)."""
import numpy as np
import pytest

from gpuvoxels_amd import _abi, engine, workloads

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (255, 1, 1), (16, 16, 1), (257, 1, 1), (19, 27, 1), (40, 40, 25)]   # 1 to 40,000 voxels (two launches)
KEYS = ("pos", "orient", "lin_mom", "ang_mom", "flags", "tfac", "init_pos", "strain", "max_strain", "small_angle")


def models():
    ms = [workloads.slab(*n, steps=0, collisions=False) for n in SIZES]
    for m in ms:   # lift off the floor, so that the first steps change only what falls
        m.ijk = m.ijk + np.array([0, 0, 2], np.int32)
    return ms


def admit(ms, precision):
    b = engine.Batch(precision=precision)
    return b, [b.admit(m) for m in ms]


@pytest.mark.parametrize("precision", [_abi.PREC_F64, _abi.PREC_F32])
def test_read_state(precision):
    ms = models()
    b, slots = admit(ms, precision)
    real = np.float64 if precision == _abi.PREC_F64 else np.float32
    for m, s in zip(ms, slots):
        nl = max(len(engine.topology(m)[0]), 1)
        x = b.read_state(s, nl=nl)
        lattice = m.ijk * m.voxel_size
        assert np.array_equal(x["pos"], lattice.astype(real).astype(np.float64))
        assert np.array_equal(x["init_pos"], lattice)
        assert np.array_equal(x["orient"], np.tile([1.0, 0, 0, 0], (m.n_voxels, 1)))
        assert not x["lin_mom"].any() and not x["ang_mom"].any() and not x["strain"].any() and not x["max_strain"].any()
        assert x["tfac"].shape == (m.n_voxels,) and x["flags"].shape == (m.n_voxels,)
    b.step(25)
    got = [b.read_state(s, nl=max(len(engine.topology(m)[0]), 1)) for m, s in zip(ms, slots)]
    st = b.poll()
    for m, s, x in zip(ms, slots, got):
        alone, (t,) = admit([m], precision)
        alone.step(25)
        y = alone.read_state(t, nl=max(len(engine.topology(m)[0]), 1))
        for k in KEYS:
            assert np.array_equal(x[k], y[k]), k
        alone.close()
        d = x["pos"] - x["init_pos"]
        dist = np.sqrt(d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1] + d[:, 2] * d[:, 2])
        assert st[s].num_measured_voxel == m.n_voxels
        assert st[s].total_distance_of_all_voxels == np.cumsum(dist)[-1]
    b.close()
