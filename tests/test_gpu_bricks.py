"""Brick copies built on the device: every brick layout reads the values the
linear grid holds, at grids smaller than a brick, whole bricks and one past,
and after the volume of a context changes in place.

The layouts share their arithmetic, so their images are the same bits."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from helpers import oracle_render, oracle_scene, xrp_scene

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 75.0), (130.0, 100.0)]


def _grid(shape, seed):
    return np.random.default_rng(seed).random(shape, dtype=np.float32)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 5), (4, 4, 4), (5, 3, 4), (8, 9, 7),
                                   (17, 16, 33)])
def test_brick_layouts_hold_the_grid(ctx, monkeypatch, shape):
    sc = xrp_scene(None, None, voxels=_grid(shape, 3))
    imgs = {}
    for layout in ("linear", "brick4", "pair", "quad", "quad_slide"):
        monkeypatch.setenv("XRP_VOXEL_LAYOUT", layout)
        imgs[layout], _ = X.render(ctx, sc, ANGLES, 24, 0.05, integrator="simple")
    sc.close()
    for layout, img in imgs.items():
        assert np.array_equal(img, imgs["linear"]), layout
    osc = oracle_scene(None, None, _grid(shape, 3))
    ref = oracle_render(osc, ANGLES, 24, 0.05, integrator="simple")
    assert float(np.abs(imgs["quad_slide"].astype(np.float64) - ref).max()) <= 1e-5


def test_volume_projections_follow_every_call(ctx):
    """Values changed in the caller's array, another array, other dimensions
    and back: each call renders what it was given."""
    cams = [X.camera_from_angles(a, p, 4.0) + (40.0, 4.0) for a, p in ANGLES]
    a, b, c = _grid((9, 12, 10), 1), _grid((9, 12, 10), 2), _grid((6, 5, 7), 3)
    for vol in (a, b, c, a, c):
        for change in (False, True):
            if change:
                vol[:3] *= 0.5
            got = X.render_volume_projections(ctx, vol, cams, 24, 0.05)
            sc = xrp_scene(None, None, voxels=vol)
            want, _ = X.render(ctx, sc, ANGLES, 24, 0.05, integrator="simple")
            sc.close()
            assert np.array_equal(got, want)
