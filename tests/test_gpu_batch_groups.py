"""Batches whose jobs take the interval march and the general guarded march side
by side, under each integrator: a group each, equal to the per-scene renders;
and a batch's general groups where XRP_INTERVALS=0 (read when it is created)
takes the interval march away."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import oracle_render, oracle_scene, xrp_scene
from test_gpu_reach import DEFORMATIONS

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 70.0), (200.0, 120.0)]


def _jobs():
    """(object, deformation, resolution, step) in turn taken by the interval
    march and refused by it."""
    coll = W.random_scene(3, max_prims=12)[0]
    lat = W.lattice(resolution=40, n_views=2)
    gyr = W.gyroid_lattice(resolution=16, n_views=1, cells=3)
    narrow = {"type": "object_collection", "objects": [
        {"type": "gyroid", "center": [0.0, 0.1, 0.0], "scale": 0.05, "thickness": 0.3, "rho": 0.4},
        {"type": "sphere", "center": [0.1, 0.0, 0.0], "radius": 0.3, "rho": 0.5}]}
    return [(W.csg().obj, None, 36, 0.01), (gyr.obj, W.TANH_SHEAR, 33, 0.008),
            (lat.obj, lat.deformation, 40, 0.004), (coll, DEFORMATIONS["sigmoid"], 24, 0.01),
            (coll, DEFORMATIONS["gaussian"], 25, 0.01), (narrow, None, 31, 0.01)]


@pytest.mark.parametrize("intervals", [True, False])
def test_interval_and_general_groups(ctx, monkeypatch, intervals):
    jobs = _jobs()
    scenes = [xrp_scene(o, d) for o, d, _, _ in jobs]
    items = [(sc, ANGLES, res, ds, {"integrator": integ, "flat_field": 0.1})
             for integ in ("simple", "hierarchical")
             for sc, (_, _, res, ds) in zip(scenes, jobs)]
    if not intervals:
        monkeypatch.setenv("XRP_INTERVALS", "0")
    b = X.Batch(ctx, items)
    single = [X.render(ctx, *it[:4], **it[4]) for it in items]
    monkeypatch.delenv("XRP_INTERVALS", raising=False)
    for rep in range(3):
        st = b.run()
        assert st["launches"] == (4 if intervals else 2)
        for k in range(len(items)):
            assert np.array_equal(b.read(k), single[k][0]), (rep, k)
    assert st["samples"] == sum(s["samples"] for _, s in single)
    for k, it in enumerate(items):
        o, d, res, ds = jobs[k % len(jobs)]
        ref = oracle_render(oracle_scene(o, d, flat_field=0.1), ANGLES, res, ds,
                            integrator=it[4]["integrator"])
        assert float(np.abs(single[k][0].astype(np.float64) - ref).max()) <= 1e-5, k
    b.close()
    for sc in scenes:
        sc.close()
