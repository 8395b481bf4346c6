"""Gyroid lattices whose cells are short against the coarse step: the
hierarchical integrator leaves them to the general march (api.cpp gyroid_plan),
which is then the faster one.

Which ran shows in the counts, which are the general march's (XRP_GYROID=0, read
per render) only where it did; the images are the same bits either way."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import oracle_render, oracle_scene, xrp_scene
from test_gpu_reach import DEFORMATIONS

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 90.0), (133.0, 61.0)]


@pytest.mark.parametrize("name,steps", [(None, 1.0), ("tanh", 1.0), ("sigmoid", 8.0)])
def test_cells_short_against_the_coarse_step(ctx, monkeypatch, name, steps):
    integ = "hierarchical"
    cells, dfm = 5, {None: None, "tanh": W.TANH_SHEAR}.get(name, DEFORMATIONS.get(name))
    obj = W.gyroid_lattice(resolution=16, n_views=1, cells=cells).obj
    obj["uc"]["objects"]["objects"][0]["thickness"] = 0.5
    sc = xrp_scene(obj, dfm)
    for ratio, takes in ((0.99 * steps, False), (1.01 * steps, True)):
        ds = 1.0 / cells / ratio
        a, sa = X.render(ctx, sc, ANGLES, 40, ds, integrator=integ, precision="guarded")
        monkeypatch.setenv("XRP_GYROID", "0")
        b, sb = X.render(ctx, sc, ANGLES, 40, ds, integrator=integ, precision="guarded")
        monkeypatch.delenv("XRP_GYROID")
        assert np.array_equal(a, b)
        same = all(sa[k] == sb[k] for k in ("reevaluated", "skipped_samples"))
        assert same != takes, (ratio, sa["skipped_samples"], sb["skipped_samples"])
        ref = oracle_render(oracle_scene(obj, dfm), ANGLES, 40, ds, integrator=integ)
        assert float(np.abs(a.astype(np.float64) - ref).max()) <= 1e-5
    sc.close()
