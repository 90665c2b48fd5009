"""A mesh collider's triangles by planes: made for a search that decides its
rows by them, and not before."""
import ctypes

import numpy as np
import pytest

import model3d_amd as m3
from model3d_amd import _lib
from oracle.binding import oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu


def _free():
    """Free device memory, asked of the HIP runtime that the library links:
    its symbols are found through the library, and no second runtime (torch
    brings its own) comes into the process."""
    L = _lib.lib()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert L.hipDeviceSynchronize() == 0
    assert L.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_planes_only_for_rows():
    """50 k triangles (6 MB of linear forms): a tree that holds the collider
    and a grid of long edges look up points; the planes come with the
    collider's own search, and its mesh is the oracle's all along."""
    mesh = m3.MarchingCubesSearch(m3.Sphere((0.03, -0.02, 0.01), 1.0), 0.0274, 4)
    n = len(mesh.faces)
    col = m3.NewColliderSolid(m3.MeshToCollider(mesh))
    tree = m3.JoinedSolid([col, m3.Sphere((0.9, 0.0, 0.0), 0.3)])
    print(f"collider of {n} triangles", flush=True)
    assert n > 48_000
    d = 0.08
    want_tree, _ = oracle_search(tree, d, 3, threads=8)
    want, _ = oracle_search(col, d, 3, threads=8)
    # the row kernels on another collider (their code, a graph's memory), then
    # all that this one is asked before its own search
    box = m3.NewColliderSolid(m3.MeshToCollider(m3.NewMeshRect((0, 0, 0), (1, 1, 1))))
    m3.MarchingCubesSearch(box, d, 3)
    for _ in range(2):
        assert same_triangles(m3.MarchingCubesSearch(tree, d, 3).triangles(), want_tree)
        m3.MarchingCubesSearch(col, 0.3, 0)
    before = _free()
    assert same_triangles(m3.MarchingCubesSearch(col, d, 3).triangles(), want)
    planes = before - _free()
    print(f"planes {planes} bytes", flush=True)
    assert planes >= 128 * n
    assert same_triangles(m3.MarchingCubesSearch(tree, d, 3).triangles(), want_tree)
    assert same_triangles(m3.MarchingCubesSearch(col, d, 3).triangles(), want)


@pytest.mark.parametrize("per_triangle", [112, 1000])
def test_planes_without_memory(per_triangle):
    """Where the planes do not fit (the forms, 128 bytes a triangle; their
    records, 104, do) the search looks its corners up: the same mesh, and no
    error of that allocation left for the calls after it."""
    mesh = m3.MarchingCubesSearch(m3.Sphere((0.01, 0.02, -0.04), 1.0), 0.0134, 4)
    n = len(mesh.faces)
    with_planes = m3.NewColliderSolid(m3.MeshToCollider(mesh))
    without = m3.NewColliderSolid(m3.MeshToCollider(mesh))
    print(f"collider of {n} triangles, {per_triangle} bytes a triangle", flush=True)
    d = 0.04
    want = m3.MarchingCubesSearch(with_planes, d, 6)
    L = _lib.lib()
    L.mc3d_selftest_alloc_cap(per_triangle * n * 5 // 4 + 4096)
    try:
        got = m3.MarchingCubesSearch(without, d, 6)
    finally:
        L.mc3d_selftest_alloc_cap(0)
    assert np.array_equal(got.vertices, want.vertices) and np.array_equal(got.faces, want.faces)
    for c in (without, with_planes):
        got = m3.MarchingCubesSearch(c, d, 6)
        assert np.array_equal(got.vertices, want.vertices) and np.array_equal(got.faces, want.faces)
