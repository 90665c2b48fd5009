"""A collider's vertices past the halvings that its triangles' bounds can decide:
the rest are lookups, a lane a vertex."""
import numpy as np
import pytest

import model3d_amd as m3
from oracle.binding import oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu


def _mesh(delta):
    s = m3.JoinedSolid([m3.Sphere((0.02, 0.01, -0.03), 0.8), m3.Capsule((-0.9, 0.1, 0.2), (0.9, 0.3, -0.4), 0.3)])
    mesh = m3.MarchingCubesSearch(s, delta, 6)
    mesh.vertices = mesh.vertices @ np.array([[0.8, -0.6, 0.0], [0.48, 0.64, -0.6], [0.36, 0.48, 0.8]])
    return mesh


# 30 .. 45 halvings: the last round by bounds, some of the rest, most of it
@pytest.mark.parametrize("iters", [30, 35, 36, 37, 41, 45, 64])
@pytest.mark.parametrize("far", [0.0, 300.0])
def test_rest_parity(iters, far):
    mesh = _mesh(0.09)
    mesh.vertices = mesh.vertices + far
    s = m3.NewColliderSolid(m3.MeshToCollider(mesh))
    print(f"ray halvings {iters} at {far}", flush=True)
    want, _ = oracle_search(s, 0.07, iters, threads=8)
    got, interior = m3.MarchingCubesInterior(s, 0.07, iters)
    assert same_triangles(got.triangles(), want)
    assert same_triangles(m3.MarchingCubesSearch(s, 0.07, iters, cull=False).triangles(), want)
    assert np.all(np.abs(interior - got.vertices).max(1) <= 0.07 / 2**iters + 1e-12 * (1 + far))


def test_rest_takes_no_longer_than_lookups():
    """290 k vertices, 60 halvings: the collider's own search against one that
    looks up every point (a tree of the collider and a ball beside it)."""
    col = m3.NewColliderSolid(m3.MeshToCollider(_mesh(0.05)))
    tree = m3.JoinedSolid([col, m3.Sphere((0.0, 0.0, 0.0), 0.05)])

    def best(s):
        return min(m3.MarchingCubesSearch(s, 0.0075, 60).stats["ms_device"] for _ in range(5))

    rows, points = best(col), best(tree)
    print(f"by rows {rows:.2f} ms, by points {points:.2f} ms", flush=True)
    assert rows < points
