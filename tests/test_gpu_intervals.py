"""The interval march (scenes of convex primitives and wide gyroids under
affine maps): audited sample by sample in FP64, against the FP64 oracle and
against the sampling marches (XRP_INTERVALS=0, read per render), over the
tree forms, map kinds, sizes and edges its rule admits.

Tolerances: audit compares every density, so it must count no difference.
The two marches add the same densities, a run of n equal terms as one product
instead of n additions: the sums differ by a few FP64 ulps and the float32
images by one rounding at most (transmittance <= 1: 6e-8)."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import load_scene_file, oracle_render, oracle_scene, xrp_scene

pytestmark = pytest.mark.gpu

ULP = 6.0e-8
AXES = [(0.0, 90.0), (90.0, 90.0), (37.0, 64.0), (180.0, 90.0)]
AFFINE = {"type": "affine", "matrix": [[1.2, 0.15, -0.1], [-0.2, 0.9, 0.25], [0.1, -0.15, 1.1]]}
CHAIN = {"type": "composed", "deformations": [
    {"type": "rigid", "displacements": [0.05, -0.1, 0.02]},
    {"type": "linear", "strains": [-0.1, 0.06, 0.0, 0.05, 0.02, -0.04]}]}


def _coll(*objs, **kw):
    return dict({"type": "object_collection", "objects": list(objs)}, **kw)


def _sphere(c, r, rho):
    return {"type": "sphere", "center": c, "radius": r, "rho": rho}


def _box(c, s, rho):
    return {"type": "box", "center": c, "sides": s, "rho": rho}


def _cyl(p0, p1, r, rho):
    return {"type": "cylinder", "p0": p0, "p1": p1, "radius": r, "rho": rho}


PPED = {"type": "parallelepiped", "origin": [-0.3, -0.2, -0.25], "v0": [0.5, 0.1, 0.0],
        "v1": [-0.1, 0.4, 0.1], "v2": [0.0, -0.1, 0.45], "rho": 0.7}
# faces, axes and cell faces that axis-aligned views meet exactly or edge-on
TIES = _coll(_box([0.0, 0.0, 0.0], [1.0, 1.0, 1.0], 1.0), _cyl([-0.6, 0.0, 0.0], [0.6, 0.0, 0.0],
                                                               0.15, -1.0),
             _box([0.25, 0.0, 0.0], [0.5, 0.5, 0.5], -0.25), _sphere([0.0, 0.0, 0.5], 0.25, 0.5))


def _many(n, seed):
    rng = np.random.default_rng(seed)
    objs = []
    for k in range(n):
        c = rng.uniform(-0.4, 0.4, 3).tolist()
        if k % 4 == 0:
            objs.append(_sphere(c, float(rng.uniform(0.02, 0.2)), float(rng.uniform(-1, 1))))
        elif k % 4 == 1:
            objs.append(_box(c, rng.uniform(0.02, 0.3, 3).tolist(), float(rng.uniform(-1, 1))))
        elif k % 4 == 2:
            objs.append(_cyl(c, (np.array(c) + rng.normal(0, 0.15, 3)).tolist(),
                             float(rng.uniform(0.01, 0.1)), float(rng.uniform(-1, 1))))
        else:
            objs.append({"type": "gyroid", "center": c, "scale": float(rng.uniform(1.0, 8.0)),
                         "thickness": float(rng.uniform(0.02, 0.3)),
                         "rho": float(rng.uniform(-1, 1))})
    return _coll(*objs)


def _tess(objs, cell, lo, hi, off=(0.0, 0.0, 0.0)):
    uc, t = {"objects": _coll(*objs)}, {"type": "tessellated_obj_coll"}
    for a, k in zip("xyz", range(3)):
        uc[a + "min"], uc[a + "max"] = off[k], off[k] + cell
        t[a + "min"], t[a + "max"] = lo, hi
    t["uc"] = uc
    return t


STRUTS = [_cyl([0.0, 0.0, 0.0], [0.25, 0.25, 0.25], 0.03, 1.0),
          _cyl([0.25, 0.0, 0.0], [0.0, 0.25, 0.25], 0.03, 0.6),
          _sphere([0.125, 0.125, 0.125], 0.06, -0.5), _box([0.0, 0.125, 0.1], [0.1, 0.1, 0.05], 0.8)]

SCENES = {
    "sphere": (_sphere([0.1, 0.0, -0.1], 0.4, 2.5), None),  # no clamp outside a collection
    "pped": (PPED, AFFINE),
    "box_negative": (_box([0.0, 0.0, 0.0], [0.4, 0.6, 0.2], -0.5), None),
    "wide_gyroid": ({"type": "gyroid", "center": [0.0, 0.1, 0.0], "scale": 0.5,
                     "thickness": 0.2, "rho": 0.3}, None),
    "ties": (TIES, None),
    "ties_affine": (TIES, AFFINE),
    "greedy": (_coll(_sphere([0.0, 0.0, 0.0], 0.3, -0.4), _box([0.1, 0.0, 0.0], [0.5, 0.4, 0.3], 0.6),
                     PPED, _sphere([0.0, 0.2, 0.0], 0.25, 0.9), greedy_dens_eval=True), None),
    "no_density": (_coll(_sphere([0.0, 0.0, 0.0], 0.3, 0.0), _box([0.0, 0.0, 0.0], [0.2, 0.2, 0.2],
                                                                 0.5)), None),
    "coll40": (_many(40, 1), CHAIN),
    "coll180": (_many(180, 2), None),
    "coll300": (_many(300, 3), AFFINE),  # past the culled list and the slots
    "struts": (_tess(STRUTS, 0.25, -0.5, 0.5), CHAIN),
    "struts_seams": (_tess(STRUTS, 0.25, -0.5, 0.5), None),  # a face in the central column
    "struts_cut": (_tess(STRUTS, 0.25, -0.43, 0.37, (0.05, -0.02, 0.11)), None),
}


def _render(ctx, monkeypatch, sc, angles, res, ds, march, **kw):
    if march == "sampling":
        monkeypatch.setenv("XRP_INTERVALS", "0")
    img, st = X.render(ctx, sc, angles, res, ds, **kw)
    monkeypatch.delenv("XRP_INTERVALS", raising=False)
    return img, st


@pytest.mark.parametrize("integ", ["simple", "hierarchical"])
@pytest.mark.parametrize("name", sorted(SCENES))
def test_intervals_match_oracle_and_sampling_march(ctx, monkeypatch, name, integ):
    obj, dfm = SCENES[name]
    sc = xrp_scene(obj, dfm)
    res, ds = (40, 0.004) if integ == "simple" else (40, 0.02)
    kw = dict(integrator=integ, flat_field=0.1, density_multiplier=1.3)
    a, sa = _render(ctx, monkeypatch, sc, AXES, res, ds, "intervals", audit=True, **kw)
    b, sb = _render(ctx, monkeypatch, sc, AXES, res, ds, "intervals", **kw)
    c, s3 = _render(ctx, monkeypatch, sc, AXES, res, ds, "sampling", **kw)
    sc.close()
    print(f"{name} {integ}: reevaluated {sb['reevaluated']}, differing pixels "
          f"{int(np.count_nonzero(b != c))}", flush=True)
    assert sa["audit_mismatch"] == 0
    assert np.array_equal(a, b)
    for key in ("samples", "skipped_samples", "fine_samples"):
        assert sa[key] == sb[key], key
    assert sb["samples"] == s3["samples"] and sb["fine_samples"] == s3["fine_samples"]
    assert float(np.abs(b.astype(np.float64) - c).max()) <= ULP
    ref = oracle_render(oracle_scene(obj, dfm, flat_field=0.1, density_multiplier=1.3), AXES, res,
                        ds, integrator=integ)
    assert float(np.abs(b.astype(np.float64) - ref).max()) <= 1e-5


@pytest.mark.parametrize("res,views,ds", [(1, 1, 0.01), (7, 3, 0.05), (65, 2, 0.5), (64, 2, 2e-5)])
def test_intervals_sizes_and_steps(ctx, monkeypatch, res, views, ds):
    """One pixel, ragged tiles, steps longer than the objects and the finest
    the rule admits."""
    for obj in (TIES, _tess(STRUTS, 0.25, -0.5, 0.5)):
        sc = xrp_scene(obj)
        for integ in ("simple", "hierarchical"):
            d = 10 * ds if integ == "hierarchical" and ds < 1e-3 else ds
            b, sb = _render(ctx, monkeypatch, sc, AXES[:views], res, d, "intervals",
                            integrator=integ)
            c, s3 = _render(ctx, monkeypatch, sc, AXES[:views], res, d, "sampling",
                            integrator=integ)
            assert sb["samples"] == s3["samples"] and sb["fine_samples"] == s3["fine_samples"]
            assert float(np.abs(b.astype(np.float64) - c).max()) <= ULP, (integ, d)
        sc.close()


@pytest.mark.parametrize("name", ["csg", "lattice"])
def test_intervals_two_passes(ctx, monkeypatch, name):
    """Large simple jobs leave the indices that need FP64 to a second pass;
    a redo list too short (XRP_REDO_CAP) renders the job again in one."""
    w = {"csg": lambda: W.csg(resolution=1024, n_views=3),
         "lattice": lambda: W.lattice(resolution=1024, n_views=3, ds=0.004)}[name]()
    images = []
    for cap in (None, "1"):
        sc = xrp_scene(w.obj, w.deformation)
        if cap:
            monkeypatch.setenv("XRP_REDO_CAP", cap)
        img, st = X.render(ctx, sc, w.angles, 1024, w.ds)
        monkeypatch.delenv("XRP_REDO_CAP", raising=False)
        print(f"{name} cap {cap}: two_pass {st['two_pass']} redo {st['redo_rays']}", flush=True)
        assert st["two_pass"] == (0 if cap else 1) and (cap or st["redo_rays"] > 0)
        images.append(img)
        sc.close()
    sc = xrp_scene(w.obj, w.deformation)
    ref, _ = _render(ctx, monkeypatch, sc, w.angles, 1024, w.ds, "sampling")
    sc.close()
    for img in images:
        assert float(np.abs(img.astype(np.float64) - ref).max()) <= ULP


def test_intervals_bytes(ctx, monkeypatch):
    obj, numbers, _ = load_scene_file("pillar_array.json")
    sc = xrp_scene(obj, numbers=numbers)
    kw = dict(output="gray8_alpha8", transparency=True, integrator="hierarchical")
    a, _ = _render(ctx, monkeypatch, sc, AXES, 96, 0.01, "intervals", **kw)
    b, _ = _render(ctx, monkeypatch, sc, AXES, 96, 0.01, "sampling", **kw)
    sc.close()
    assert np.array_equal(a, b)
