"""GroupTriangles with the axes sorted one by one, as for more triangles than
one sort takes: the same order as the oracle's, on meshes small enough to test."""
import numpy as np
import pytest

import model3d_amd as m3
from model3d_amd import _lib
from oracle.binding import oracle_group_triangles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 1024, 1025, 5003, 40_000])
def test_group_three_sorts(n):
    rng = np.random.default_rng(n)
    tris = (np.round(rng.uniform(-1, 1, (n, 1, 3)) * 16) / 16 + rng.uniform(-0.02, 0.02, (n, 3, 3))).reshape(n, 9)
    v = np.ascontiguousarray(tris.reshape(-1, 3))
    f = np.arange(3 * n, dtype=np.uint32)
    perm = np.empty(n, dtype=np.uint32)
    print(f"group by three sorts {n}", flush=True)
    L = _lib.lib()
    _lib.check(L.mc3d_selftest_group_sorts(_lib.context(0), v.ctypes.data, len(v), f.ctypes.data, n, perm.ctypes.data))
    assert np.array_equal(perm, oracle_group_triangles(tris))
    assert np.array_equal(perm, m3.group_order(tris))
