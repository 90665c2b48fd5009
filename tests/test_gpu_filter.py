"""The device's block filter (all leaves of MarchingCubesFilter's recursion
asked at once) against the host recursion that asks the same collider block
by block through a callback: the meshes are equal where leaves are decided
in each of its ways -- by the tables, by the open list, past the open list,
at the root, and for blocks too long to gather."""
import numpy as np
import pytest

import model3d_amd as m3
from tests.helpers import same_triangles

pytestmark = pytest.mark.gpu


def _csg():
    return m3.SubtractedSolid(m3.JoinedSolid([m3.Sphere((0.0, 0.0, 0.0), 0.6), m3.Capsule((0.2, 0.3, 0.0), (0.9, 0.5, 0.4), 0.2)]),
                              m3.Cylinder((-0.8, 0.0, 0.1), (0.5, 0.1, 0.0), 0.25))


def _box(mn, mx):
    return m3.Rect(mn, mx), m3.NewMeshRect(mn, mx)


def _cases():
    flat, flat_mesh = _box((0.0, 0.0, 0.0), (1.0, 1.0, 0.02))
    rod, rod_mesh = _box((0.0, 0.0, 0.0), (4.0, 0.03, 0.02))
    dot, dot_mesh = _box((0.0, 0.0, 0.0), (0.04, 0.03, 0.05))
    part = _csg()
    fine = m3.MarchingCubesSearch(part, 0.05, 4)
    half = m3.Mesh.from_triangles(fine.triangles()[: len(fine.faces) // 2])
    return {
        # every leaf lies on a face of twelve large triangles: more open
        # leaves than the list holds
        "flat": (flat, flat_mesh, 0.004),
        # blocks much longer than a word
        "rod": (rod, rod_mesh, 0.01),
        # the root is a leaf
        "dot": (dot, dot_mesh, 0.02),
        # many small triangles (the tables), and a mesh that covers half
        "part": (part, fine, 0.03),
        "half": (part, half, 0.021),
        # a collider off to one side, and one that touches nothing
        "aside": (part, m3.NewMeshRect((0.5, -0.2, -0.3), (3.0, 0.7, 0.3)), 0.025),
        "apart": (part, m3.NewMeshRect((5.0, 5.0, 5.0), (6.0, 6.0, 6.0)), 0.04),
    }


@pytest.mark.parametrize("name", ["flat", "rod", "dot", "part", "half", "aside", "apart"])
def test_device_filter_equals_host_recursion(name):
    solid, mesh, delta = _cases()[name]
    col = m3.MeshToCollider(mesh)
    print(f"block filter {name}", flush=True)
    got = m3.MarchingCubesSearchFilter(solid, col.RectCollision, delta, 3)
    asked = [0]

    def host(rect):
        asked[0] += 1
        return col.RectCollision(rect)

    want = m3.MarchingCubesSearchFilter(solid, host, delta, 3)
    print(f"{asked[0]} blocks asked, {len(want.faces)} triangles", flush=True)
    assert same_triangles(got.triangles(), want.triangles())
    assert (len(want.faces) > 0) == (name != "apart")
