"""The surrogate march against the network's own predictions at the samples
of its rays, for tables of which none, some or all levels are held in LDS.

With table entries that BF16 represents, the march's packed tables and the
predictions' FP32 ones hold the same values, so the densities differ only where
the sample positions' FP32 rounding (about 1e-6 of the unit cell, times up to
64 cells) moves a BF16 rounding: a few in a hundred of a sample's 96 roundings,
2^-9 each, hence about 2e-4 of a density, of either sign, and 2e-5 over the
hundred samples of a ray at step 0.01.  A level read from wrong entries is
0.05 of a density, 5e-3 of a ray.  A sample within that rounding of the
bounds may fall on either side of them: a ray's expected value is with it or
without."""
import math

import numpy as np
import pytest

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import O, xrp_scene

pytestmark = pytest.mark.gpu

TOL = 1e-3
EDGE = 1e-6  # FP32 position error
R, FOV, HALF = 4.0, 40.0, 1.74  # the march runs over [R - HALF, R + HALF]


@pytest.mark.parametrize("log2_table,n_min,n_max", [
    (4, 2, 64),    # all levels in LDS, hashed to 16 entries
    (10, 4, 64),   # all, dense and hashed
    (12, 16, 64),  # nine of 16
    (15, 8, 64),   # the dense ones among the first
    (16, 40, 64),  # none: the first level is too large
])
def test_march_is_its_predictions(ctx, log2_table, n_min, n_max):
    res, ds = 33, 0.01
    w = W.gyroid_lattice(resolution=res, n_views=1, cells=3)
    sc = xrp_scene(w.obj, None)
    sur = X.Surrogate(ctx, sc, log2_table=log2_table, n_min=n_min, n_max=n_max)
    rng = np.random.default_rng(log2_table)
    t = 1 << log2_table
    sur.set_params(X.join_surrogate_params({
        "tables": rng.integers(-64, 65, (16, t, 2)) / 128.0,
        "W1": rng.normal(0, 1 / math.sqrt(32), (32, 64)),
        "b1": rng.normal(0, 0.1, 64),
        "W2": rng.normal(0, 1 / math.sqrt(64), (64, 64)),
        "b2": rng.normal(0, 0.1, 64),
        "w3": rng.normal(0, 2 / math.sqrt(64), 64),
        "b3": np.float64(0.2),
    }))
    angles = [(17.0, 83.0), (140.0, 90.0)]
    img, _ = sur.render(angles, res, 0.5 * ds, ds, 0.0)
    s = R - HALF + (np.arange(math.ceil(2.0 * HALF / ds)) + 0.5) * ds
    pts, where = [], []
    for v, (az, polar) in enumerate(angles):
        eye, cam = O.camera_from_angles(az, polar, R)
        for i in range(res):
            for j in range(res):
                o, d = O.pixel_ray(eye, cam, res, FOV, i, j)
                p = o[None, :] + s[:, None] * (d / np.linalg.norm(d))[None, :]
                p = p[(np.abs(p) <= 0.5 + EDGE).all(axis=1)]
                pts.append(p)
                where.append(np.full(len(p), (v * res + i) * res + j))
    p, at = np.concatenate(pts), np.concatenate(where)
    u = (p - w.obj["uc"]["xmin"]) / (w.obj["uc"]["xmax"] - w.obj["uc"]["xmin"])
    dens = sur.predict((u - np.floor(u)).astype(np.float32)).astype(np.float64)
    edge = (np.abs(p) >= 0.5 - EDGE).any(axis=1)
    T, E = (np.bincount(at[m], weights=dens[m] * ds, minlength=2 * res * res)
            .reshape(2, res, res) for m in (~edge, edge))
    # two views of 48 x 48 tiles go to resident workgroups, one does not: the
    # same bits
    both, _ = sur.render(angles, 190, 0.5 * ds, ds, 0.0)
    for v in range(2):
        one, _ = sur.render(angles[v:v + 1], 190, 0.5 * ds, ds, 0.0)
        assert np.array_equal(one[0], both[v])
    sur.close()
    err = np.minimum(np.abs(img - np.exp(-T)), np.abs(img - np.exp(-(T + E))))
    print(f"{int(edge.sum())} samples at the bounds", flush=True)
    print(f"2^{log2_table}: max {err.max():.2e} mean {err.mean():.2e}", flush=True)
    assert err.max() <= TOL
