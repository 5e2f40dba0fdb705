"""The tile planner with bodies at the far ends of the lattice's index range, on the CPU: the same
invariants, the same blocks as with the bodies close together, and no work or memory for the
empty space between."""
import subprocess

import numpy as np
import pytest

from test_tile_plan import checker  # noqa: F401


def blobs(distance, order):
    """Three separate 9 x 9 x 9 cubes `distance` apart along one axis, voxels shuffled or not."""
    z, y, x = np.meshgrid(*(np.arange(9),) * 3, indexing="ij")
    one = np.stack([x.ravel(), y.ravel(), z.ravel()], 1).astype(np.int64)
    cells = np.concatenate([one + [(i - 1) * distance, 0, 0] for i in range(3)])
    if order:
        cells = np.random.default_rng(order).permutation(cells)
    at = {tuple(c): i for i, c in enumerate(cells.tolist())}
    links = []
    for c, i in at.items():
        for a in range(3):
            d = list(c)
            d[a] += 1
            if tuple(d) in at:
                links.append((i, at[tuple(d)], a))
    return cells, links


def plan(checker, cells, links):  # noqa: F811
    lines = ["%d %d 300 400 256" % (len(cells), len(links))]
    lines += ["%d %d %d" % tuple(r) for r in cells] + ["%d %d %d" % r for r in links]
    r = subprocess.run([checker], input="\n".join(lines) + "\n", stdout=subprocess.PIPE, text=True, check=True, timeout=60)
    return r.stdout.split()


@pytest.mark.parametrize("order", [0, 5])
def test_far_apart(checker, order):  # noqa: F811
    near = plan(checker, *blobs(20, order))
    assert near[0] == "ok", near
    for distance in (1 << 20, 1 << 30, (1 << 31) - 20):
        assert plan(checker, *blobs(distance, order)) == near
