"""Batches of scenes that take next to no time a ray: the work queue's own
atomics were most of a launch, and the interval march's form, with more waves,
took up to 1.7 times the sampling march's time."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from helpers import xrp_scene

pytestmark = pytest.mark.gpu

SPHERE = {"type": "object_collection", "objects": [
    {"type": "sphere", "center": [0.1, 0.0, -0.1], "radius": 0.2, "rho": 1.0}]}


def _batch(ctx, items, repeats=5):
    b = X.Batch(ctx, items)
    st = min((b.run() for _ in range(repeats)), key=lambda s: s["kernel_ms"])
    got = [b.read(k) for k in range(len(items))]
    b.close()
    return st, got


@pytest.mark.parametrize("integ", ["simple", "hierarchical"])
@pytest.mark.parametrize("scenes,views,res", [(1, 8, 256), (1, 2, 64), (6, 3, 200), (1, 1, 8),
                                              (2, 1, 17)])
def test_simple_scenes_cost_no_more_than_the_sampling_march(ctx, monkeypatch, scenes, views, res,
                                                            integ):
    sc = [xrp_scene(SPHERE) for _ in range(scenes)]
    angles = [(20.0 + 50 * k, 70.0 + 5 * k) for k in range(views)]
    items = [(s, angles, res, 0.05, {"integrator": integ}) for s in sc]
    a, got = _batch(ctx, items)
    monkeypatch.setenv("XRP_INTERVALS", "0")
    b, ref = _batch(ctx, items)
    monkeypatch.delenv("XRP_INTERVALS")
    one, st = X.render(ctx, sc[0], angles, res, 0.05, integrator=integ)
    for s in sc:
        s.close()
    print(f"{scenes} x {views} x {res}^2 {integ}: {1e3 * a['kernel_ms']:.0f} us, sampling "
          f"{1e3 * b['kernel_ms']:.0f}", flush=True)
    for x, y in zip(got, ref):
        assert np.array_equal(x, one)
        assert float(np.abs(x.astype(np.float64) - y).max()) <= 6.0e-8
    # counts are added by runs of items and come out whole
    assert a["samples"] == b["samples"] == scenes * st["samples"]
    assert a["kernel_ms"] < 1.3 * b["kernel_ms"]
