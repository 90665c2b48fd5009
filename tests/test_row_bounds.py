"""How much the row form of an atom leaves open (mc3d_selftest_line, on the
host): every open corner is evaluated on its own, and an edge with many open
points is halved point by point, so lines that real parts have many of must be
decided."""
import ctypes

import numpy as np
import pytest

import model3d_amd as m3
from model3d_amd import _lib
from model3d_amd.solids import LibBackend


def _line(s, p, axis, h, levels):
    """(open points, points inside) of a line; wrong certainties fail."""
    b = LibBackend()
    hs = s._build(b)
    sure, maybe, inside = ctypes.c_uint64(), ctypes.c_uint64(), ctypes.c_uint64()
    try:
        _lib.check(_lib.lib().mc3d_selftest_line(hs, (ctypes.c_double * 3)(*p), axis, h, levels, ctypes.byref(sure), ctypes.byref(maybe),
                                                 ctypes.byref(inside)))
    finally:
        b.release(hs)
        b.close()
    n = (1 << levels) if levels else 64
    mask = (1 << n) - 1
    assert sure.value & ~inside.value & mask == 0 and inside.value & ~maybe.value & mask == 0
    return bin(maybe.value & ~sure.value & mask).count("1"), bin(inside.value & mask).count("1")


def _unit(axis, v=1.0):
    return tuple(v if a == axis else 0.0 for a in range(3))


@pytest.mark.parametrize("kind", [m3.Cylinder, m3.Capsule])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_lines_in_a_cap_plane(kind, axis):
    """A part's end faces lie in planes of the grid (which begins at its
    bounds): rows and edges in them are decided but for the round side."""
    rng = np.random.default_rng(axis)
    worst = inside = 0
    for _ in range(200):
        base = [float(v) for v in rng.uniform(-2, 2, 3)]
        length, r = float(rng.uniform(0.1, 2)), float(rng.uniform(0.1, 0.5))
        tip = [b + (length if a == axis else 0.0) for a, b in enumerate(base)]
        s = kind(base, tip, r)
        for k in range(3):
            if k == axis:
                continue
            o = 3 - k - axis
            p = [0.0, 0.0, 0.0]
            p[axis] = (base, tip)[int(rng.integers(2))][axis]
            p[o] = base[o] + float(rng.uniform(-0.9, 0.9)) * r
            for levels in (0, 6):
                h = 0.02 if levels == 0 else 2.5 * r
                p[k] = base[k] - float(rng.uniform(1.1, 1.2)) * r
                opened, n = _line(s, p, k, h, levels)
                worst, inside = max(worst, opened), inside + n
    assert inside > 4000
    assert worst <= 2


@pytest.mark.parametrize("kind", ["sphere", "cylinder", "capsule"])
@pytest.mark.parametrize("far", [0.0, 1e3, 1e4, 1e5, 1e6])
def test_lines_far_from_the_origin(kind, far):
    """A solid's place costs its bounds nothing: rows and edges (spacing 0.01)
    through solids of size one leave on average less than one point open, up to
    10^8 spacings from the origin."""
    rng = np.random.default_rng(int(far) + len(kind))
    opened = inside = 0
    lines = 400
    for _ in range(lines):
        c = [far + float(v) for v in rng.uniform(-1, 1, 3)]
        d = rng.normal(size=3)
        d /= np.linalg.norm(d)
        e = [a + float(b) for a, b in zip(c, d)]
        s = m3.Sphere(c, 0.5) if kind == "sphere" else (m3.Cylinder if kind == "cylinder" else m3.Capsule)(c, e, 0.4)
        k, levels = int(rng.integers(3)), (0, 6)[int(rng.integers(2))]
        t = float(rng.uniform(0.1, 0.9)) if kind != "sphere" else 0.0
        p = [a + t * (b - a) + float(rng.uniform(-0.2, 0.2)) for a, b in zip(c, e)]
        p[k] -= float(rng.uniform(0.0, 0.8))
        o, n = _line(s, p, k, 0.01 if levels == 0 else 0.8, levels)
        opened, inside = opened + o, inside + n
    assert inside > 10 * lines
    assert opened < lines
