"""Stitching of z slabs at the edges of its forms: tiles of 1024 vertices whose
counts are summed or (past 2048 of them) scanned, slabs without a vertex,
planes without one, a slab per cube layer.  The stitched mesh is the whole
grid's, so every comparison is exact."""
import numpy as np
import pytest

import model3d_amd as m3

pytestmark = pytest.mark.gpu


def _vertex_codes(v):
    """A 64-bit code per vertex (of its bits; -0 is not produced here)."""
    u = np.ascontiguousarray(v).view(np.uint64)
    h = np.zeros(len(u), np.uint64)
    for c, k in enumerate((0x9E3779B97F4A7C15, 0xC2B2AE3D27D4EB4F, 0x165667B19E3779F9)):
        h += (u[:, c] ^ (u[:, c] >> np.uint64(29))) * np.uint64(k)
    return h ^ (h >> np.uint64(31))


def _same(whole, got):
    a, b = _vertex_codes(whole.vertices), _vertex_codes(got.vertices)
    assert len(a) == len(b) and np.array_equal(np.sort(a), np.sort(b))
    # a triangle's code does not depend on which corner comes first
    mix = lambda h, f: (h[f] * np.uint64(3) + h[np.roll(f, 1, 1)] * np.uint64(5) * h[f]).sum(1)
    assert np.array_equal(np.sort(mix(a, whole.faces)), np.sort(mix(b, got.faces)))


@pytest.mark.parametrize("planes", [1, 2, 7, 21, 100])
def test_slabs_with_empty_planes(planes):
    # two spheres apart in z: slabs and shared planes without a vertex between
    s = m3.JoinedSolid([m3.Sphere((0, 0, -2), 0.5), m3.Sphere((0.1, 0, 2), 0.4)])
    print(f"slabs of two spheres, planes={planes}", flush=True)
    _same(m3.MarchingCubesSearch(s, 0.05, 8), m3.MarchingCubesSearch(s, 0.05, 8, slab_planes=planes))


# vertices of the second slab about 1024 n, its tiles partly filled, and more than 2048 tiles
@pytest.mark.parametrize("delta,planes", [(0.11, 3), (0.06, 5), (0.0015, 400)])
def test_slab_tiles(delta, planes):
    s = m3.Sphere((0, 0, 0), 1.0)
    print(f"slabs of a sphere, delta={delta}", flush=True)
    whole = m3.MarchingCubesSearch(s, delta, 4)
    got = m3.MarchingCubesSearch(s, delta, 4, slab_planes=planes)
    if delta == 0.0015:
        assert len(whole.vertices) > 2 * 2_200_000
    _same(whole, got)
