"""Solids whose atoms are all untransformed spheres, boxes, capsules and
cylinders are meshed by rows (a lane decides the corners of a word, or the
midpoints of an edge, from the interval on which each atom is true): the
meshes are the oracle's bit for bit where those intervals are hardest --
surfaces through corners, along rows and grazing them, words of every fill,
bricks of every shape, deep programs."""
import numpy as np
import pytest

import model3d_amd as m3
from oracle.binding import oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu

FP64 = m3.MC3D_PREC_FP64
GUARD = m3.MC3D_PREC_FP32_GUARD


def _deep(n, at=0.0):
    """A balanced tree of 2^n overlapping spheres (n + 1 stack entries)."""
    if n == 0:
        return m3.Sphere((at, 0.1 * at, -0.2 * at), 0.5)
    a, b = _deep(n - 1, at - 0.3 / 2**n), _deep(n - 1, at + 0.3 / 2**n)
    return m3.IntersectedSolid([a, b]) if n % 2 else m3.JoinedSolid([a, m3.SubtractedSolid(b, m3.Sphere((at, 0.4, 0.1), 0.2))])


def _solids():
    x, y, z = (1.0, 0.0, 0.0), (0.0, 1.0, 0.0), (0.0, 0.0, 1.0)

    def neg(v):
        return tuple(-c for c in v)

    return {
        # cylinders and capsules along each axis, through the origin
        "aligned": (m3.JoinedSolid([m3.Cylinder(neg(x), x, 0.25), m3.Capsule(neg(y), y, 0.25), m3.Cylinder(z, neg(z), 0.125)]),
                    0.0625),
        # faces, axes and end caps on the corners of a power-of-two grid
        "on_corners": (m3.SubtractedSolid(m3.Rect((-1.0, -0.75, -0.5), (1.0, 0.75, 0.5)),
                                          m3.JoinedSolid([m3.Cylinder((0.0, 0.0, -1.0), (0.0, 0.0, 1.0), 0.25),
                                                          m3.Sphere((0.5, 0.5, 0.5), 0.25)])), 0.03125),
        # a surface much larger than the grid, nearly flat in it
        "huge": (m3.ClipSolid(m3.Sphere((0.0, 0.0, -300.0), 300.0), (-1.0, -1.0, -0.5), (1.0, 1.0, 0.25)), 0.03),
        # far from the origin, thin
        "far": (m3.JoinedSolid([m3.Capsule((1000.0, 1000.0, 999.0), (1000.9, 1000.01, 999.0), 0.05),
                                m3.Rect((1000.2, 999.9, 998.9), (1000.5, 1000.1, 999.1))]), 0.02),
        # a point-like capsule (a zero-length segment), a radius of zero
        "degenerate": (m3.JoinedSolid([m3.Capsule((0.0, 0.0, 0.0), (0.0, 0.0, 0.0), 0.3), m3.Sphere((0.1, 0.2, 0.0), 0.0),
                                       m3.Sphere((0.3, 0.0, 0.1), 0.2)]), 0.04),
        "deep": (_deep(5), 0.03),
    }


@pytest.mark.parametrize("name", list(_solids()))
@pytest.mark.parametrize("iters", [0, 6, 13])
def test_rows_parity(name, iters):
    s, delta = _solids()[name]
    print(f"rows parity {name} iters={iters}", flush=True)
    want, _ = oracle_search(s, delta, iters, threads=8)
    assert len(want) > 0
    for kw in (dict(brick=0), dict(brick=8, precision=FP64), dict(brick=3), dict(brick=16, precision=FP64), dict(cull=False)):
        got = m3.MarchingCubesSearch(s, delta, iters, **kw)
        assert same_triangles(got.triangles(), want), kw


@pytest.mark.parametrize("nx", [3, 63, 64, 65, 128, 129])
def test_rows_word_fill(nx):
    """Rows that end anywhere in a word, in a batch of two solids."""
    delta = 1.0 / (nx - 2.5)
    a = m3.Cylinder((0.0, 0.2, 0.1), (1.0, 0.25, 0.15), 0.11)
    b = m3.ClipSolid(m3.JoinedSolid([m3.Sphere((0.3, 0.2, 0.0), 0.3), m3.Capsule((0.1, 0.1, 0.1), (0.9, 0.3, 0.2), 0.1)]),
                     (0.0, 0.0, -0.2), (1.0, 0.4, 0.3))
    print(f"rows word fill nx={nx}", flush=True)
    for cull in (True, False):
        got = m3.MarchingCubesSearchBatch([a, b], [delta, delta], [5, 7], cull=cull)
        for s, it, m in zip((a, b), (5, 7), got):
            want, _ = oracle_search(s, delta, it, threads=8)
            assert same_triangles(m.triangles(), want)


def test_rows_statistics_runs_agree():
    """A statistics run decides point by point; its mesh is the same."""
    s, delta = _solids()["aligned"]
    print("rows against points", flush=True)
    for precision in (FP64, GUARD):
        a = m3.MarchingCubesSearch(s, delta, 8, precision=precision)
        b = m3.MarchingCubesSearch(s, delta, 8, precision=precision, count_mismatch=True)
        assert np.array_equal(a.vertices, b.vertices) and np.array_equal(a.faces, b.faces)
        assert b.stats["corner_flops64"] > 0 and b.stats["guard_violations"] == 0
