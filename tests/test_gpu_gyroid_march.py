"""The gyroid march (gyroid_march.hpp) against the general march of the same
scene (XRP_GYROID=0, read per render): the same bits, samples and fine samples
for every deformation kind, in one pass and in two, both output formats, and
no audit mismatch; and scenes it must leave alone."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import oracle_render, oracle_scene, xrp_scene
from test_gpu_reach import DEFORMATIONS

pytestmark = pytest.mark.gpu

TOL = 1e-5
DEFS = dict(DEFORMATIONS, straight=None)
for _src in "xyz":
    for _axis in "xyz":
        if _src != _axis:
            DEFS[f"tanh {_src}{_axis}"] = {"type": "tanh_shear", "amplitude": -0.07, "rate": 6.0,
                                           "source": _src, "direction": _axis}

# cells, centre, thickness, rho, resolution, ds
SCENES = [
    (6, [0.0, 0.0, 0.0], 0.1, 1.0, 64, 0.002),
    (3, [0.03, -0.05, 0.011], 0.45, 0.6, 67, 0.0071),
    (1, [0.2, 0.1, 0.0], 0.9, 2.5, 33, 0.03),   # above 1: a cell does not clamp it
    (2, [0.0, 0.0, 0.0], 1e-3, 1.0, 65, 0.004),  # thinner than a fine step
    (4, [0.0, 0.0, 0.0], 0.3, 1.0, 7, 0.9),     # steps larger than a cell
]


def _object(cells, centre, thickness, rho):
    w = W.gyroid_lattice(resolution=16, n_views=1, cells=cells)
    w.obj["uc"]["objects"]["objects"][0].update(center=centre, thickness=thickness, rho=rho)
    return w.obj


def _both(ctx, monkeypatch, sc, res, ds, integ, **kw):
    angles = [(20.0, 90.0), (0.0, 90.0), (133.0, 61.0)]
    out = []
    for on in ("1", "0"):
        monkeypatch.setenv("XRP_GYROID", on)
        out += X.render(ctx, sc, angles, res, ds, integrator=integ, precision="guarded", **kw)
    return angles, out


@pytest.mark.parametrize("integ", ["simple", "hierarchical"])
@pytest.mark.parametrize("scene", range(len(SCENES)))
@pytest.mark.parametrize("name", list(DEFS))
def test_gyroid_march_is_the_general_march(ctx, monkeypatch, name, scene, integ):
    *what, res, ds = SCENES[scene]
    obj = _object(*what)
    sc = xrp_scene(obj, DEFS[name])
    angles, (a, sa, b, sb) = _both(ctx, monkeypatch, sc, res, ds, integ)
    assert np.array_equal(a, b)
    assert sa["samples"] == sb["samples"] and sa["fine_samples"] == sb["fine_samples"]
    # in two passes, and with every ray's list cut to nothing
    monkeypatch.setenv("XRP_TWO_PASS", "1")
    for most in ("14", "0"):
        monkeypatch.setenv("XRP_DEFER_MAX", most)
        _, (c, st, _, _) = _both(ctx, monkeypatch, sc, res, ds, integ)
        assert st["two_pass"] == 1 and np.array_equal(c, b)
        assert st["samples"] == sb["samples"] and st["fine_samples"] == sb["fine_samples"]
    monkeypatch.delenv("XRP_TWO_PASS")
    _, (_, st, _, _) = _both(ctx, monkeypatch, sc, res, ds, integ, audit=True)
    assert st["audit_mismatch"] == 0
    sc.close()
    if res < 64:
        ref = oracle_render(oracle_scene(obj, DEFS[name]), angles, res, ds, integrator=integ)
        assert float(np.max(np.abs(a.astype(np.float64) - ref))) <= TOL


def _two_gyroids(obj):
    kids = obj["uc"]["objects"]["objects"]
    kids.append(dict(kids[0], thickness=0.2, rho=0.5))


def _part_period(obj):
    obj["uc"]["objects"]["objects"][0]["scale"] *= 0.9


def _negative_scale(obj):
    obj["uc"]["objects"]["objects"][0]["scale"] *= -1.0


def _long_cells(obj):
    # whole periods that differ per axis
    obj["uc"]["xmax"] *= 2.0
    obj["uc"]["xmin"] *= 2.0


@pytest.mark.parametrize("integ", ["simple", "hierarchical"])
@pytest.mark.parametrize("change", [_two_gyroids, _part_period, _negative_scale, _long_cells])
def test_gyroid_march_other_forms(ctx, monkeypatch, change, integ):
    obj = _object(4, [0.0, 0.0, 0.0], 0.3, 1.0)
    change(obj)
    sc = xrp_scene(obj, W.TANH_SHEAR)
    angles, (a, sa, b, sb) = _both(ctx, monkeypatch, sc, 40, 0.01, integ)
    sc.close()
    assert np.array_equal(a, b)
    assert sa["samples"] == sb["samples"] and sa["fine_samples"] == sb["fine_samples"]
    ref = oracle_render(oracle_scene(obj, W.TANH_SHEAR), angles, 40, 0.01, integrator=integ)
    assert float(np.max(np.abs(a.astype(np.float64) - ref))) <= TOL
