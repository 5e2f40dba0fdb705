"""Tiled simulations on the kernel with the links of all axes at once (taken when one launch
holds their finer tiles and nothing else shares the chip) against the per-step kernels: the
same bits, sampling steps and short launches included; and the way there and back as other
simulations join and leave between calls."""
import numpy as np
import pytest

from gpuvoxels_amd import _abi, engine, workloads
from gpuvoxels_amd.model import MT

pytestmark = pytest.mark.gpu

KEYS = ("pos", "orient", "lin_mom", "ang_mom", "flags", "tfac", "strain", "max_strain", "small_angle")


def robot(seed, grid):
    m = workloads.robot(np.random.default_rng(seed), grid=grid, steps=0)
    m.materials[1].fixed = seed % 2
    m.materials[2].mat_model, m.materials[2].fail_stress = _abi.MDL_LINEAR_FAIL, 800.0
    return m


def state(b, slots, models):
    st = b.poll()
    return [(b.read_state(s, nl=len(engine.topology(m)[0])), st[s]) for s, m in zip(slots, models)]


def same(a, c):
    for (x, sx), (y, sy) in zip(a, c):
        assert sx.steps == sy.steps and sx.state == sy.state and sx.current_time == sy.current_time
        for k in KEYS:
            assert np.array_equal(x[k], y[k], equal_nan=True), k


# two tiles; plans of 448 slots; as large as the shape takes; too many for one launch
@pytest.mark.parametrize("precision", [_abi.PREC_F64, _abi.PREC_F32])
@pytest.mark.parametrize("grids", [[14], [15, 27], [44, 44], [40, 40, 41, 42]])
def test_equals_step_kernels(precision, grids):
    models = [robot(i, g) for i, g in enumerate(grids)]
    got = []
    for noalloc in (False, True):
        b = engine.Batch(precision=precision, path=_abi.PATH_AUTO, steps_per_launch=70)
        slots = [b.admit(m) for m in models]
        for n in (1, 2, 150):
            (b.step_noalloc if noalloc else b.step)(n)
        got.append(state(b, slots, models))
        b.close()
    same(*got)


@pytest.mark.parametrize("precision", [_abi.PREC_F64, _abi.PREC_F32])
def test_others_join_and_leave(precision):
    big, small, plate = robot(3, 20), robot(4, 8), workloads.slab(20, 20, 2, steps=0)
    more = [robot(5 + i, 43) for i in range(3)]
    b = engine.Batch(precision=precision, path=_abi.PATH_AUTO)
    s = b.admit(big)
    b.step(20)                                  # finer tiles
    fine = b.workgroups(s)
    t = b.admit(small)
    b.step(20)                                  # beside a one-workgroup simulation
    coarse = b.workgroups(s)
    assert 1 < coarse < fine
    b.retire(t)
    u = b.admit(plate)
    b.step(20)                                  # beside the per-step kernels
    assert b.workgroups(s) == coarse
    b.retire(u)
    b.step(20)
    assert b.workgroups(s) == fine
    v = [b.admit(m) for m in more]
    b.step(20)                                  # larger tiles again, of either kernel
    assert b.workgroups(s) < fine
    for x in v:
        b.retire(x)
    b.step(20)
    assert b.workgroups(s) == fine
    c = engine.Batch(precision=precision, path=_abi.PATH_AUTO)
    r = c.admit(big)
    c.step_noalloc(120)
    same(state(b, [s], [big]), state(c, [r], [big]))
    b.close()
    c.close()


def test_plans_are_kept_as_others_leave():
    """Simulations planned among others go on as the tiles they have when some leave (a plan takes
    longer than it would save), and one that has had plans of both sizes goes back to the smaller."""
    models = [robot(20 + i, 40) for i in range(3)]
    b = engine.Batch(precision=_abi.PREC_F32, path=_abi.PATH_AUTO)
    s = [b.admit(models[0])]
    b.step(10)
    alone = b.workgroups(s[0])
    s += [b.admit(m) for m in models[1:]]
    b.step(10)
    among = [b.workgroups(x) for x in s]
    assert 1 < among[0] < alone
    b.retire(s[2])
    b.step(10)
    assert [b.workgroups(x) for x in s[:2]] == [alone, among[1]]
    got = state(b, s[:2], models[:2])
    b.close()
    for i, n in ((0, 30), (1, 20)):
        c = engine.Batch(precision=_abi.PREC_F32, path=_abi.PATH_STREAM)
        r = c.admit(models[i])
        c.step_noalloc(n)
        same([got[i]], state(c, [r], [models[i]]))
        c.close()


@pytest.mark.parametrize("precision", [_abi.PREC_F64, _abi.PREC_F32])
def test_divergence_and_stop(precision):
    """Simulations flung apart (large-angle links, then a diverged one: the launch is run again up
    to that step), stopped by their step budget within a launch, and by a condition."""
    def models():
        ms = [robot(30 + i, 17) for i in range(3)]
        rng = np.random.default_rng(8)
        ms[0].init_velocity = rng.normal(0, 300.0, (ms[0].n_voxels, 3))
        ms[1].init_velocity = rng.normal(0, 3.0, (ms[1].n_voxels, 3))
        ms[1].max_steps = 77
        ms[2].stop_tokens = [(MT["mtCONST"], 0.001), (MT["mtVAR"], 4.0), (MT["mtGREATERTHAN"], 0.0), (MT["mtEND"], 0.0)]
        return ms
    got = []
    for noalloc in (False, True):
        ms = models()
        b = engine.Batch(precision=precision, path=_abi.PATH_AUTO, steps_per_launch=60)
        s = [b.admit(m) for m in ms]
        (b.step_noalloc if noalloc else b.step)(150)
        if not noalloc:
            assert all(b.workgroups(x) > 1 for x in s)
        got.append(state(b, s, ms))
        b.close()
    assert [x[1].state for x in got[0]] == [_abi.SIM_DIVERGED, _abi.SIM_DONE, _abi.SIM_DONE]
    assert np.any(got[0][1][0]["small_angle"] == 0)
    same(*got)
