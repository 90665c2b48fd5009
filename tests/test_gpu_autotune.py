"""The autotuner times each shape that can differ once: solids with a row form
have only bricks to choose from."""
import pytest

import model3d_amd as m3
from model3d_amd import autotune

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solid,shapes", [(m3.Sphere((0, 0, 0), 0.5), 3), (m3.Torus((0, 0, 0), (0, 0, 1), 0.5, 0.2), 3 * 3 * 3)])
def test_candidates(solid, shapes):
    print(f"autotune {solid}", flush=True)
    best = autotune.tune(solid, 0.05, 4, reps=1)
    assert len(best["table"]) == shapes
    assert len({tuple(r[k] for k in ("brick", "rows_per_walk", "waves_per_brick")) for r in best["table"]}) == shapes
    assert best["ms"] == min(r["ms"] for r in best["table"])
