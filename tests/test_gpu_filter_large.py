"""The block filter where most leaves are open: large triangles, whose corners
lie in few leaves (the blocks above a hit leaf are asked of the triangle that
hits it), and grids of more leaves than are asked at a time."""
import time

import numpy as np
import pytest

import model3d_amd as m3
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu


def _solid():
    return m3.SubtractedSolid(m3.JoinedSolid([m3.Sphere((0.0, 0.0, 0.0), 0.9), m3.Capsule((0.2, 0.3, 0.0), (0.9, 0.5, 0.4), 0.3)]),
                              m3.Cylinder((-0.8, 0.0, 0.1), (0.5, 0.1, 0.0), 0.25))


def _soup(n, size, kind=""):
    r = np.random.default_rng(n)
    if n == 1:
        return m3.MeshCollider(np.array([[[-1.1, -0.9, 0.3], [1.2, -0.8, -0.2], [0.1, 1.3, 0.1]]]))
    t = r.uniform(-1, 1, (n, 1, 3)) + r.uniform(-size, size, (n, 3, 3))
    if kind == "degenerate":  # needles and points
        t[::3, 2] = t[::3, 1]
        t[::5, 1] = t[::5, 2] = t[::5, 0]
    if kind == "flat":  # in planes of the blocks' faces
        t[:, :, 0] = np.round(t[:, :1, 0] * 8) / 8
    return m3.MeshCollider(t)


@pytest.mark.parametrize("n,size,kind", [(1, 1.0, ""), (12, 1.0, ""), (60, 1.0, "flat"), (300, 1.0, "degenerate"), (300, 0.5, ""),
                                         (3000, 0.3, "degenerate"), (3000, 0.05, "")])
def test_large_triangles(n, size, kind):
    col, s = _soup(n, size, kind), _solid()
    print(f"block filter of {n} triangles of {size} {kind}", flush=True)
    got = m3.MarchingCubesSearchFilter(s, col.RectCollision, 0.04, 3)
    want = m3.MarchingCubesSearchFilter(s, lambda rect: col.RectCollision(rect), 0.04, 3)
    print(f"{len(want.faces)} triangles", flush=True)
    assert len(want.faces) > 0
    assert same_triangles(got.triangles(), want.triangles())


def test_leaves_in_parts():
    """834^3 cubes: 2^23 paths of halvings, 2^22 asked at a time.  Small balls in
    every corner of a large box; coarse-to-fine finds all of each."""
    balls = [m3.Sphere((x, y, z), 0.09) for x in (-0.85, 0.8) for y in (-0.8, 0.85) for z in (-0.83, 0.84)]
    s = m3.ForceSolidBounds(m3.JoinedSolid(balls + [m3.Sphere((0.0, 0.01, 0.02), 0.1)]), (-0.999, -0.999, -0.999), (0.999, 0.999, 0.999))
    print("leaves in parts", flush=True)
    want = m3.MarchingCubesSearch(s, 0.0024, 2)
    got = m3.MarchingCubesC2F(s, 0.03, 0.0024, 0.0, 2)
    assert len(want.faces) > 100_000
    assert np.array_equal(got.vertices, want.vertices) and np.array_equal(got.faces, want.faces)


def test_large_triangles_take_little_time():
    """Twelve large triangles at 202^3 corners: a filtered call, the recursion
    included, takes less than 4 times the search alone (about 1.6 times; 8 times
    where most open leaves are asked one after another by the wave that found
    them and each block above a leaf of the whole mesh)."""
    col, s = _soup(12, 1.0), _solid()
    def best(f):
        ts = []
        for _ in range(8):
            t = time.perf_counter()
            f()
            ts.append(time.perf_counter() - t)
        return min(ts)

    whole = best(lambda: m3.MarchingCubesSearch(s, 0.01, 1))
    filtered = best(lambda: m3.MarchingCubesSearchFilter(s, col.RectCollision, 0.01, 1))
    print(f"whole {1e6 * whole:.0f} us, filtered {1e6 * filtered:.0f} us", flush=True)
    assert filtered < 4 * whole
