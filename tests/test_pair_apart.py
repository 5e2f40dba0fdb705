"""The contact loops' early test (pairApart in vx3_kernels.inl) leaves out only pairs whose
contact force is zero: its formula against pairContact's, both in numpy with the kernels'
types, at lengths within a few units in the last place of the contact distance, at tiny and
huge voxels, and with infinities and NaN."""
import numpy as np
import pytest

F = np.float32


def rel(o, tfi, tfj, nom):
    """pairContact's overlap: the contact distance minus the length."""
    b1, b2 = nom * nom.dtype.type(tfi), nom * nom.dtype.type(tfj)
    three = nom.dtype.type(3)
    dist = F(((b1 + b1 + b1) / three + (b2 + b2 + b2) / three) * nom.dtype.type(0.625))
    return dist, dist - np.sqrt(o[0] * o[0] + o[1] * o[1] + o[2] * o[2])


def apart(o, tfi, tfj, nom):
    reach = F(nom) * (tfi + tfj) * F(0.625)
    r2 = reach * reach
    return (o[0] * o[0] + o[1] * o[1] + o[2] * o[2] > r2 * (F(1) + F(2.0 ** -18))) & (r2 > F(1e-30))


@pytest.mark.parametrize("real", [np.float64, np.float32])
@pytest.mark.parametrize("size", [1e-25, 1e-20, 1e-15, 1e-6, 1e-2, 1.0, 1e6, 1e18, 1e19])
def test_only_zero_forces(real, size):
    rng = np.random.default_rng(7)
    seen = 0
    with np.errstate(all="ignore"):
        for _ in range(4000):
            nom = real(size * rng.uniform(0.5, 2))
            tfi, tfj = F(rng.uniform(0.5, 1.5)), F(rng.uniform(0.5, 1.5))
            dist, _ = rel(np.zeros(3, F), tfi, tfj, nom)
            d = rng.normal(size=3)
            d /= np.linalg.norm(d)
            far = rng.choice([1 + rng.integers(-8, 9) * 2.0 ** -24, 1 + rng.uniform(0, 2.0 ** -16), rng.uniform(0, 3)])
            o = F(d * float(dist) * far)
            a = apart(o, tfi, tfj, nom)
            seen += bool(a)
            assert not (a and rel(o, tfi, tfj, nom)[1] > 0)
            for bad in (np.nan, np.inf, -np.inf):
                q = o.copy()
                q[rng.integers(3)] = bad
                assert not (apart(q, tfi, tfj, nom) and rel(q, tfi, tfj, nom)[1] > 0)
    if 1e-12 < size < 1e18:
        assert seen > 500
