"""Volume projections of a small volume that comes again: no slower than with
the copies reused, and new values, dimensions or a failed call never render the
old volume."""
import time

import numpy as np
import pytest

import xray_projection_render_amd as X
from helpers import xrp_scene

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 75.0), (130.0, 100.0)]
CAMS = [X.camera_from_angles(a, p, 4.0) + (40.0, 4.0) for a, p in ANGLES]


def _want(ctx, vol):
    sc = xrp_scene(None, None, voxels=vol)
    img, _ = X.render(ctx, sc, ANGLES, 24, 0.05, integrator="simple")
    sc.close()
    return img


@pytest.mark.parametrize("shape", [(3, 4, 5), (40, 33, 30), (64, 64, 128), (65, 64, 128)])
def test_values_that_change_in_place(ctx, shape):
    """Up to 2 MiB (the third) and past it; the last voxel alone, the sign of a
    zero, a NaN's bits, back again, other arrays and dimensions."""
    rng = np.random.default_rng(2)
    vol = rng.random(shape, dtype=np.float32)
    other = np.ascontiguousarray(vol.transpose(2, 0, 1))  # the same bytes' size
    for change in (None, "last", "zero", None, "back", "shape"):
        if change == "last":
            vol[-1, -1, -1] += 0.5
        elif change == "zero":
            vol[:2] = -0.0
        elif change == "back":
            vol[...] = rng.random(shape, dtype=np.float32)
        v = other if change == "shape" else vol
        assert np.array_equal(X.render_volume_projections(ctx, v, CAMS, 24, 0.05), _want(ctx, v))
    assert np.array_equal(X.render_volume_projections(ctx, vol, CAMS, 24, 0.05), _want(ctx, vol))


def test_two_contexts(ctx):
    a, b = (np.random.default_rng(k).random((20, 20, 20), dtype=np.float32) for k in (1, 2))
    with X.Context(0) as second:
        for _ in range(2):
            assert np.array_equal(X.render_volume_projections(ctx, a, CAMS, 24, 0.05), _want(ctx, a))
            assert np.array_equal(X.render_volume_projections(second, b, CAMS, 24, 0.05),
                                  _want(ctx, b))


def test_the_same_volume_again_costs_less_than_a_new_one(ctx):
    """4 x 32^2 of 64 x 64 x 100 voxels: with its copies there, a call is one
    launch; copied over and rebuilt each time the two took the same."""
    vols = [np.random.default_rng(k).random((64, 64, 100), dtype=np.float32) for k in range(2)]
    t = {}
    for name, pick in (("same", lambda k: vols[0]), ("new", lambda k: vols[k % 2])):
        times = []
        for k in range(40):
            a = time.perf_counter()
            X.render_volume_projections(ctx, pick(k), CAMS, 32, 0.01)
            times.append(time.perf_counter() - a)
        t[name] = sorted(times)[10]
    print(f"same {1e6 * t['same']:.0f} us, new {1e6 * t['new']:.0f} us", flush=True)
    assert t["same"] < 0.9 * t["new"]
