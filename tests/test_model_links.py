"""The links of a model against a look-up over its voxels in plain Python: order, ends and
axes, scattered and dense voxels, negative coordinates, and
duplicates refused."""
import numpy as np
import pytest

from gpuvoxels_amd import engine, workloads

DIRS = [(1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]


def expected(ijk):
    where, neg, pos, axis = {}, [], [], []
    for v, c in enumerate(map(tuple, ijk.tolist())):
        where[c] = v
        for k, d in enumerate(DIRS):
            u = where.get(tuple(np.add(c, d).tolist()))
            if u is not None:
                neg.append(u if k % 2 else v)
                pos.append(v if k % 2 else u)
                axis.append(k // 2)
    return neg, pos, axis


@pytest.mark.parametrize("n,box,low", [(1, 1, 0), (2, 2, 5), (4, 2, -1), (40, 5, -3), (900, 13, 0), (4000, 17, -9), (300, 2000, -1000)])
def test_links(n, box, low):
    rng = np.random.default_rng(n)
    cells = np.unique(rng.integers(0, box, (4 * n, 3)), axis=0)
    ijk = (rng.permutation(cells)[:n] + low).astype(np.int32)
    m = workloads.cube(2, steps=0)
    m.ijk = ijk
    m.mat, m.phase = np.zeros(len(ijk), np.int32), np.zeros(len(ijk))
    neg, pos, axis, _ = engine.topology(m)
    assert [neg.tolist(), pos.tolist(), axis.tolist()] == list(expected(ijk))
    if len(ijk) > 1:
        m.ijk = np.concatenate([ijk[:-1], ijk[:1]])
        with pytest.raises(Exception, match="duplicate voxel"):
            engine.topology(m)
