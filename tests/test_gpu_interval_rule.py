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


def _sphere(c, r, rho):
    return {"type": "sphere", "center": list(c), "radius": float(r), "rho": rho}


def _overlapping(n):
    """Spheres that all hold the centre."""
    rng = np.random.default_rng(n)
    return {"type": "object_collection", "objects": [
        _sphere(rng.uniform(-0.05, 0.05, 3), rng.uniform(0.35, 0.45), 0.01) for _ in range(n)]}


def _shells(n):
    return {"type": "object_collection", "objects": [
        _sphere((0.0, 0.0, 0.0), 0.45 * (1 - 0.9 * k / n), 0.3 if k % 2 == 0 else -0.2)
        for k in range(n)]}


def _gyroids(n, scale):
    rng = np.random.default_rng(n)
    return {"type": "object_collection", "objects": [
        {"type": "gyroid", "center": rng.uniform(-0.5, 0.5, 3).tolist(), "scale": scale,
         "thickness": 0.3, "rho": 0.3} for _ in range(n)]}


@pytest.mark.parametrize("make,integ,ds,takes", [
    (lambda: _overlapping(60), "simple", 0.01, True),
    (lambda: _overlapping(60), "hierarchical", 0.05, True),
    (lambda: _overlapping(180), "simple", 0.01, True),
    (lambda: _overlapping(180), "hierarchical", 0.05, False),  # past 128 that overlap
    (lambda: _overlapping(250), "simple", 0.01, False),        # past the most slots
    (lambda: _shells(100), "hierarchical", 0.05, True),
    (lambda: _shells(250), "simple", 0.01, False),
    (lambda: _gyroids(24, 0.28), "simple", 0.08, True),
    (lambda: _gyroids(40, 0.28), "simple", 0.01, True),
    (lambda: _gyroids(40, 0.28), "simple", 0.08, False),       # 22 samples a period
    (lambda: _gyroids(40, 4.0), "hierarchical", 0.08, True),
])
def test_children_that_overlap(ctx, monkeypatch, make, integ, ds, takes):
    """Many children at one place: more run slots, or the sampling march."""
    obj = make()
    took, img = _takes(ctx, monkeypatch, obj, 40, ds, integ)
    assert took == takes
    ref = oracle_render(oracle_scene(obj), ANGLES, 40, ds, integrator=integ)
    assert float(np.abs(img.astype(np.float64) - ref).max()) <= 1e-5


@pytest.mark.parametrize("make,integ,ds", [
    (lambda: _overlapping(60), "hierarchical", 0.02),
    (lambda: _overlapping(180), "simple", 0.004),
    (lambda: _shells(60), "hierarchical", 0.02),
    (lambda: _gyroids(60, 4.0), "simple", 0.004),
])
def test_overlaps_are_no_slower(ctx, monkeypatch, make, integ, ds):
    """Out of run slots these took 4 to 30 times the sampling march's time; the
    test asks for less than twice."""
    sc = xrp_scene(make())
    views = [(20.0 + 17 * k, 60.0 + 5 * k) for k in range(4)]
    best = {}
    for march in ("0", "1"):
        monkeypatch.setenv("XRP_INTERVALS", march)
        best[march] = min(X.render(ctx, sc, views, 256, ds, integrator=integ)[1]["kernel_ms"]
                          for _ in range(3))
    sc.close()
    print(f"{integ} {ds}: intervals {best['1']:.2f} ms, sampling {best['0']:.2f}", flush=True)
    assert best["1"] < 2.0 * best["0"]


def test_batch_of_overlaps(ctx, monkeypatch):
    """In a batch, jobs of more slots than 96 join the sampling march's group."""
    objs = [_overlapping(60), _overlapping(150), _gyroids(60, 1.0)]
    scenes = [xrp_scene(o) for o in objs]
    items = [(sc, ANGLES, 24, 0.02, {"integrator": "simple"}) for sc in scenes]
    b = X.Batch(ctx, items)
    st = b.run()
    got = [b.read(k) for k in range(len(items))]
    b.close()
    assert st["launches"] == 2
    for k, sc in enumerate(scenes):
        ref = oracle_render(oracle_scene(objs[k]), ANGLES, 24, 0.02, integrator="simple")
        assert float(np.abs(got[k].astype(np.float64) - ref).max()) <= 1e-5, k
        sc.close()


def test_batch_keeps_scenes_of_many_gyroids(ctx):
    """A place has at most one run of each gyroid, so 60 of them fit the 96 slots
    of a batch, where the sampling march of one such scene outlasts all others."""
    objs = [_overlapping(60), _gyroids(60, 1.0)]
    scenes = [xrp_scene(o) for o in objs]
    b = X.Batch(ctx, [(sc, ANGLES, 24, 0.02, {"integrator": "simple"}) for sc in scenes])
    assert b.run()["launches"] == 1
    for k, sc in enumerate(scenes):
        ref = oracle_render(oracle_scene(objs[k]), ANGLES, 24, 0.02, integrator="simple")
        assert float(np.abs(b.read(k).astype(np.float64) - ref).max()) <= 1e-5, k
        sc.close()
    b.close()
