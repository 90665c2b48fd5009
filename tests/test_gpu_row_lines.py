"""Lines that the row forms leave open all along -- on a cylinder's side, far
from the origin, after many halvings -- which a wave decides point by point:
the meshes are the oracle's, and the halvings past the bounds' precision cost
an evaluation each."""
import pytest

import model3d_amd as m3
from oracle.binding import oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu


def _solids():
    d = 1 / 32
    # rows and edges along the sides of cylinders of a whole number of spacings, end faces in the grid's planes
    sides = m3.JoinedSolid([m3.Cylinder(tuple(-x for x in ax), ax, 8 * d) for ax in ((1.0, 0, 0), (0, 0.75, 0), (0, 0, 0.5))])
    plate = m3.SubtractedSolid(m3.Rect((-1.0, -0.5, 0.0), (1.0, 0.5, 0.25)),
                               m3.JoinedSolid([m3.Cylinder((x / 4, y / 4, 0.0), (x / 4, y / 4, 0.25), 0.125) for x in (-2, 0, 2) for y in (-1, 1)]))
    o = 3.0e6
    far = m3.JoinedSolid([m3.Sphere((o, -o, o), 0.7), m3.Cylinder((o, -o, o), (o + 1.0, 0.4 - o, o), 0.3),
                          m3.Capsule((o, -o, o - 0.2), (o - 0.9, 0.1 - o, o + 0.3), 0.25)])
    return {"sides": (sides, d), "plate": (plate, d), "far": (far, 0.0625)}


@pytest.mark.parametrize("name", list(_solids()))
@pytest.mark.parametrize("iters", [0, 8, 30, 64])
def test_open_lines(name, iters):
    s, d = _solids()[name]
    want, _ = oracle_search(s, d, iters, threads=8)
    assert len(want) > 0
    for kw in (dict(), dict(brick=8), dict(brick=3), dict(cull=False)):
        print(f"open lines {name} iters={iters} {kw}", flush=True)
        assert same_triangles(m3.MarchingCubesSearch(s, d, iters, **kw).triangles(), want), kw


def test_open_lines_in_a_batch():
    solids = [s for s, _ in _solids().values()] * 3
    deltas = [d for _, d in _solids().values()] * 3
    iters = [5, 40, 8, 64, 6, 30, 2, 9, 24]
    for cull in (True, False):
        print(f"open lines in a batch, cull={cull}", flush=True)
        for s, d, i, m in zip(solids, deltas, iters, m3.MarchingCubesSearchBatch(solids, deltas, iters, cull=cull)):
            want, _ = oracle_search(s, d, i, threads=8)
            assert same_triangles(m.triangles(), want)


def test_many_halvings_cost_their_evaluations():
    """64 halvings of one sphere against 8: less than 4 times the device time
    (about 1.4 times; 6.6 times with every open point of a bracket evaluated)."""
    s = m3.Sphere((0.1, 0.2, 0.3), 1.0)

    def best(iters):
        return min(m3.MarchingCubesSearch(s, 0.02, iters, cull=False).stats["ms_device"] for _ in range(10))

    few, many = best(8), best(64)
    print(f"8 halvings {1e3 * few:.1f} us, 64 halvings {1e3 * many:.1f} us", flush=True)
    assert many < 4 * few
