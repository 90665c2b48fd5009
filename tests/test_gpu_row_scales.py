"""Solids decided by rows at scales far from one: the meshes are the oracle's
bit for bit where squares, their rounding and the roots of both are tiny or
huge, and where a solid is small beside its distance from the origin."""
import numpy as np
import pytest

import model3d_amd as m3
from oracle.binding import oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu


def _parity(s, delta, iters, **kw):
    want, _ = oracle_search(s, delta, iters, threads=8)
    assert len(want) > 0
    got = m3.MarchingCubesSearch(s, delta, iters, **kw)
    assert same_triangles(got.triangles(), want), kw


@pytest.mark.parametrize("scale", [1e-80, 1e-30, 1e-18, 1e-16, 1e-8, 1e8, 1e60])
def test_rows_at_scale(scale):
    def at(*c):
        return tuple(x * scale for x in c)

    s = m3.SubtractedSolid(
        m3.JoinedSolid([m3.Sphere(at(0.1, -0.2, 0.05), 0.7 * scale), m3.Cylinder(at(-0.9, 0.4, -0.5), at(0.65, -0.3, 0.5), 0.35 * scale),
                        m3.Capsule(at(0.5, 0.35, 0.0), at(0.5, 1.1, 0.0), 0.25 * scale)]),
        m3.Rect(at(-0.3, -0.3, 0.1), at(0.25, 0.5, 0.8)))
    for kw in (dict(), dict(brick=8, precision=m3.MC3D_PREC_FP64), dict(cull=False)):
        print(f"rows at scale {scale} {kw}", flush=True)
        _parity(s, 0.0625 * scale, 7, **kw)


@pytest.mark.parametrize("center,r", [((1e-18, 0.7e-18, 0.3e-18), 1e-25), ((1e-18, 0.7e-18, 0.3e-18), 1e-23), ((1e8, 0.7e8, 0.3e8), 10.0)])
def test_rows_small_and_far(center, r):
    """Spheres and tilted cylinders much smaller than their coordinates."""
    end = tuple(c + d * r for c, d in zip(center, (2.1, 0.9, -1.3)))
    for s in (m3.Sphere(center, r), m3.Cylinder(center, end, r), m3.Capsule(center, end, r)):
        for kw in (dict(), dict(cull=False)):
            print(f"rows far {center} {r} {kw}", flush=True)
            _parity(s, r / 10.3, 5, **kw)
