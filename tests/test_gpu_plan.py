"""The brick plan's lists of nodes to walk, at their edges: programs of one
node, around whole blocks of 64 nodes and around the longest listed program;
bricks that meet none, some and all of a program's atoms; constants and every
operator over parts that miss.  Culling changes no corner, so the meshes are
those of the unculled grid bit for bit."""
import numpy as np
import pytest

import model3d_amd as m3
from oracle.binding import oracle_search
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu


def _pieces(n, spread, seed=3):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, (n, 3)) * spread
    r = rng.uniform(0.05, 0.2, n)
    return [m3.Sphere(tuple(p), q) if i % 3 else m3.Rect(tuple(p - q), tuple(p + q)) for i, (p, q) in enumerate(zip(c, r))]


def _mixed(parts):
    """Groups of four under each operator, joined."""
    out = []
    for i in range(0, len(parts), 4):
        g = parts[i:i + 4]
        if len(g) < 4:
            out += g
            continue
        a, b, c, d = g
        out.append(m3.SubtractedSolid(m3.JoinedSolid([a, b]), c) if i % 8 else m3.SubtractedSolid(m3.JoinedSolid([a, d]), m3.IntersectedSolid([b, c])))
    return m3.JoinedSolid(out) if len(out) > 1 else out[0]


@pytest.mark.parametrize("brick", [0, 2, 8])
@pytest.mark.parametrize("n", [1, 2, 16, 17, 32, 33, 64, 65, 129])
def test_plan_lists(n, brick):
    s = _mixed(_pieces(n, 1.0))
    print(f"plan of {n} atoms, brick={brick}", flush=True)
    want, _ = oracle_search(s, 0.06, 4, threads=8)
    assert same_triangles(m3.MarchingCubesSearch(s, 0.06, 4, brick=brick).triangles(), want)


# 2 n - 1 nodes: 16383 are listed, 16385 and more are not
@pytest.mark.parametrize("n", [8192, 8193])
def test_plan_longest_list(n):
    s = m3.JoinedSolid(_pieces(n, 4.0))
    print(f"plan of {n} atoms", flush=True)
    culled = m3.MarchingCubesSearch(s, 0.25, 2)
    whole = m3.MarchingCubesSearch(s, 0.25, 2, cull=False)
    assert len(culled.vertices) > 1000
    assert same_triangles(culled.triangles(), whole.triangles())


def test_plan_of_several_solids():
    ss = [_mixed(_pieces(n, 1.0, n)) for n in (1, 33, 64, 5, 130)]
    print("plan of 5 solids", flush=True)
    for s, m in zip(ss, m3.MarchingCubesSearchBatch(ss, 0.06, 4)):
        want, _ = oracle_search(s, 0.06, 4, threads=8)
        assert same_triangles(m.triangles(), want)
