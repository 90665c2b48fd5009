"""A collider's corners by rows (k_rays.hip) at its edges: rows of every word
fill and past one wave's 1024 corners, slabs that end within a wave's rows,
meshes of a few large and of many small triangles, coarse grids whose rows'
planes lie further apart than the bins, faces and edges on the grid's corners,
rays that graze faces.  Every corner is the oracle's, so the meshes are equal
bit for bit."""
import numpy as np
import pytest

import model3d_amd as m3
from oracle.binding import oracle_contains, oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu

D = np.array([0.5224892708603626, 0.10494477243214506, 0.43558938446126527])


def _box_tris(lo, hi):
    c = np.array([[(lo, hi)[i >> k & 1][k] for k in range(3)] for i in range(8)], float)
    quads = [(0, 2, 3, 1), (4, 5, 7, 6), (0, 1, 5, 4), (2, 6, 7, 3), (0, 4, 6, 2), (1, 3, 7, 5)]
    return np.array([c[[q[0], q[i], q[i + 1]]] for q in quads for i in (1, 2)])


def _turned(tris, axis, angle):
    a = np.array(axis, float) / np.linalg.norm(axis)
    k = np.array([[0, -a[2], a[1]], [a[2], 0, -a[0]], [-a[1], a[0], 0]])
    return tris @ (np.eye(3) + np.sin(angle) * k + (1 - np.cos(angle)) * k @ k).T


def _along_ray(t):
    """t with its z edges along the ray: four of a box's faces graze it."""
    z = D / np.linalg.norm(D)
    x = np.cross([0.0, 1.0, 0.0], z)
    x /= np.linalg.norm(x)
    return t @ np.stack([x, np.cross(z, x), z])


def _blob(delta):
    s = m3.SubtractedSolid(m3.JoinedSolid([m3.Sphere((0, 0, 0), 0.8), m3.Capsule((-0.9, 0.1, 0.2), (0.9, 0.3, -0.4), 0.3)]),
                           m3.Sphere((0.3, 0.2, 0.5), 0.4))
    return _turned(oracle_search(s, delta, 6, threads=8)[0].reshape(-1, 3, 3), (1, 2, 3), 0.7)


def _two():
    return np.concatenate([_box_tris((-1, -0.5, -0.25), (0.5, 0.5, 0.5)), _box_tris((0.0, -0.25, 0.0), (1.0, 0.25, 1.0))])


MESHES = {
    "box": lambda: _box_tris((-1, -0.75, -0.5), (1, 0.75, 0.5)),
    "boxes": _two,
    "turned": lambda: _turned(_two(), (3, -1, 2), 1.1),
    "grazed": lambda: _along_ray(_box_tris((-0.4, -0.3, -0.8), (0.4, 0.3, 0.8))),
    "blob": lambda: _blob(0.08),
    "fine": lambda: _blob(0.03),
    "one": lambda: np.array([[[-0.5, -0.5, 0.0], [0.5, -0.4, 0.1], [0.1, 0.6, 0.9]]]),
}


@pytest.mark.parametrize("name", list(MESHES))
@pytest.mark.parametrize("delta,cull", [(0.0625, False), (0.25, True), (0.031, True), (0.7, False)])
def test_ray_rows_parity(name, delta, cull):
    s = m3.NewColliderSolid(m3.MeshToCollider(MESHES[name]()))
    print(f"ray rows {name} delta={delta}", flush=True)
    want, _ = oracle_search(s, delta, 5, threads=8)
    assert same_triangles(m3.MarchingCubesSearch(s, delta, 5, cull=cull).triangles(), want)


@pytest.mark.parametrize("nx", [30, 31, 32, 33, 63, 64, 65, 1022, 1023, 1024, 1025, 1057, 2049])
def test_ray_rows_widths(nx):
    # a bar along x, so that a row has about nx corners
    tris = _turned(_box_tris((0, 0, 0), (nx - 2.5, 5.3, 4.2)), (0.2, 1, 0.1), 0.0007)
    s = m3.NewColliderSolid(m3.MeshToCollider(tris))
    print(f"ray rows of {nx} corners", flush=True)
    want, _ = oracle_search(s, 1.0, 3, threads=8)
    assert len(want) > 0
    assert same_triangles(m3.MarchingCubesSearch(s, 1.0, 3).triangles(), want)


@pytest.mark.parametrize("planes", [1, 3, 6])
def test_ray_rows_slabs(planes):
    s = m3.NewColliderSolid(m3.MeshToCollider(_blob(0.08)))
    print(f"ray rows in slabs of {planes}", flush=True)
    want, _ = oracle_search(s, 0.05, 5, threads=8)
    assert same_triangles(m3.MarchingCubesSearch(s, 0.05, 5, slab_planes=planes).triangles(), want)


@pytest.mark.parametrize("iters", [0, 1, 2, 5, 6, 7, 8, 13, 30, 60])
@pytest.mark.parametrize("name", ["boxes", "turned", "blob"])
def test_ray_bisection(name, iters):
    s = m3.NewColliderSolid(m3.MeshToCollider(MESHES[name]()))
    print(f"ray bisection {name} iters={iters}", flush=True)
    want, _ = oracle_search(s, 0.11, iters, threads=8)
    assert same_triangles(m3.MarchingCubesSearch(s, 0.11, iters).triangles(), want)
    mesh, interior = m3.MarchingCubesInterior(s, 0.11, iters)
    assert same_triangles(mesh.triangles(), want)
    assert np.all(oracle_contains(s, interior))
