"""Device GroupTriangles (model3d/bvh.go:118-156) at the edges of its forms:
nodes of LDS size, the tiles of a partition, tile counts that are summed or
scanned, equal midpoints, NaN boxes.  The order is a fixed function of the
input (equal midpoints in index order), so every comparison is exact."""
import numpy as np
import pytest

import model3d_amd as m3
from oracle.binding import oracle_group_triangles

pytestmark = pytest.mark.gpu


def _triangles(n, kind, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, (n, 1, 3))
    if kind == "ties":  # a few distinct midpoints per axis
        c = np.round(c * 4) / 4
    t = c + rng.uniform(-0.02, 0.02, (n, 3, 3)) * (kind != "ties")
    if kind == "nan":
        t[rng.random((n, 3, 3)) < 0.02] = np.nan
    return t.reshape(n, 9)


@pytest.mark.parametrize("kind", ["random", "ties", "nan"])
@pytest.mark.parametrize("n", [1, 2, 3, 64, 65, 341, 342, 682, 683, 1023, 1024, 1025, 1366, 2047, 2048, 2049, 4097, 20011])
def test_group_sizes(n, kind):
    tris = _triangles(n, kind, n)
    print(f"group {n} {kind}", flush=True)
    assert np.array_equal(m3.group_order(tris), oracle_group_triangles(tris))


# past 2048 tiles of 1024 entries the counts are scanned: 3 n of them at the
# split of the sorted keys, n of them at a level's partition
@pytest.mark.parametrize("n", [699_050, 699_051, 2_097_153])
def test_group_scanned_tiles(n):
    tris = _triangles(n, "random", 1)
    print(f"group {n}", flush=True)
    assert np.array_equal(m3.group_order(tris), oracle_group_triangles(tris))
