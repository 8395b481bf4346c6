"""Scenes that the interval march leaves to the sampling marches because it
would be the slower one (api.cpp line_plan), and those it takes, on either side
of its rules.

Which march ran shows in the counts: the interval march settles all samples but
one per change of density, the sampling march (XRP_INTERVALS=0, read per render)
those within its safe radius.  A scene left alone gives the same image and
counts with the switch and without."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from helpers import oracle_render, oracle_scene, xrp_scene

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 80.0), (131.0, 60.0)]
COUNTS = ("samples", "reevaluated", "skipped_samples", "fine_samples")


def _takes(ctx, monkeypatch, obj, res, ds, integ, views=ANGLES):
    """Whether the interval march ran; images within one FP32 neighbour."""
    sc = xrp_scene(obj)
    kw = dict(integrator=integ)
    a, sa = X.render(ctx, sc, views, res, ds, **kw)
    monkeypatch.setenv("XRP_INTERVALS", "0")
    b, sb = X.render(ctx, sc, views, res, ds, **kw)
    monkeypatch.delenv("XRP_INTERVALS")
    sc.close()
    assert float(np.abs(a.astype(np.float64) - b).max()) <= 6.0e-8
    same = [sa[k] == sb[k] for k in COUNTS]
    assert sa["samples"] == sb["samples"] and sa["fine_samples"] == sb["fine_samples"]
    if all(same):
        assert np.array_equal(a, b)
    return not all(same), a


def _cells(n, sides):
    rng = np.random.default_rng(n)
    side = min(sides)
    objs = []
    for k in range(n):
        c = (rng.uniform(0.2, 0.8, 3) * np.array(sides)).tolist()
        objs.append({"type": "sphere", "center": c, "radius": 0.15 * side, "rho": 0.5} if k % 2 == 0
                    else {"type": "box", "center": c, "sides": [0.2 * side] * 3, "rho": 0.7})
    t = {"type": "tessellated_obj_coll",
         "uc": {"objects": {"type": "object_collection", "objects": objs}}}
    for a, s in zip("xyz", sides):
        t["uc"][a + "min"], t["uc"][a + "max"] = 0.0, s
        t[a + "min"], t[a + "max"] = -0.5, 0.5
    return t


@pytest.mark.parametrize("integ,least", [("simple", 6.0), ("hierarchical", 24.0)])
@pytest.mark.parametrize("n", [1, 24])
@pytest.mark.parametrize("sides", [(0.25, 0.25, 0.25), (0.25, 0.125, 0.2)])
def test_cells_short_against_the_step(ctx, monkeypatch, sides, n, integ, least):
    """Cells of fewer indices than the rule asks for along the shortest side."""
    obj = _cells(n, sides)
    for indices, takes in ((1.0, False), (0.99 * least, False), (1.01 * least, True)):
        unit = min(sides) / indices
        ds = 10 * unit if integ == "hierarchical" else unit
        took, img = _takes(ctx, monkeypatch, obj, 24, ds, integ)
        assert took == takes, indices
        ref = oracle_render(oracle_scene(obj), ANGLES, 24, ds, integrator=integ)
        assert float(np.abs(img.astype(np.float64) - ref).max()) <= 1e-5
