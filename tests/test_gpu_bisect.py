"""Bisection of solids without a row form (cones, tori, frames), a lane a
vertex or eight lanes a vertex: every count of halvings modulo the three that
are decided at once, meshes on both sides of the line between the two forms,
interior points, bricks of one program and of several in a wave, no culling."""
import numpy as np
import pytest

import model3d_amd as m3
from oracle.binding import oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu

GUARD, FP64 = m3.MC3D_PREC_FP32_GUARD, m3.MC3D_PREC_FP64


def _solid():
    return m3.SubtractedSolid(
        m3.JoinedSolid([m3.Torus((0.1, 0.0, 0.0), (0.0, 0.0, 1.0), 0.6, 0.2), m3.Cone((0.2, 0.1, 0.9), (-0.3, 0.0, -0.6), 0.5),
                        m3.Sphere((-0.5, 0.4, 0.1), 0.3)]),
        m3.Cylinder((-1.0, 0.0, 0.1), (1.0, 0.3, 0.0), 0.15))


@pytest.mark.parametrize("precision", [GUARD, FP64])
@pytest.mark.parametrize("iters", [0, 1, 2, 3, 4, 5, 6, 7, 8, 17])
def test_bisect_spread_halvings(iters, precision):
    s = _solid()
    print(f"bisect iters={iters}", flush=True)
    want, _ = oracle_search(s, 0.06, iters, threads=8)
    assert same_triangles(m3.MarchingCubesSearch(s, 0.06, iters, precision=precision).triangles(), want)
    whole = m3.MarchingCubesSearch(s, 0.06, iters, precision=precision, cull=False)
    assert same_triangles(whole.triangles(), want)


# 47 k and 50 k vertices: either side of 48 k (49,152)
@pytest.mark.parametrize("delta", [0.016, 0.0155])
def test_bisect_spread_line(delta):
    s = _solid()
    mesh = m3.MarchingCubesSearch(s, delta, 7)
    print(f"bisect of {len(mesh.vertices)} vertices", flush=True)
    want, _ = oracle_search(s, delta, 7, threads=8)
    assert same_triangles(mesh.triangles(), want)


def test_bisect_spread_interior():
    s = _solid()
    from oracle.binding import oracle_contains
    print("bisect interior", flush=True)
    mesh, interior = m3.MarchingCubesInterior(s, 0.05, 7)
    assert np.all(oracle_contains(s, interior))
    whole = m3.MarchingCubesSearch(s, 0.05, 7)
    assert np.array_equal(mesh.vertices, whole.vertices)
