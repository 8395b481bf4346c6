"""FP64 marches of a voxel root, from the quad bricks and (without allocation,
where no quads are resident) from the linear copy: the same bits, and the
oracle's images; grids smaller than a brick, whole bricks and one past, with
empty regions for the hierarchical march's toggles."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from helpers import oracle_render, oracle_scene, xrp_scene

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 75.0), (130.0, 100.0)]
DEFORM = {
    "none": None,
    "affine": {"type": "affine", "matrix": [[1.9, 0.1, 0.0], [0.0, 2.0, -0.2], [0.1, 0.0, 2.1]]},
    "sigmoid": {"type": "sigmoid", "amplitude": 0.1, "center": 0.1, "lengthscale": 0.2,
                "direction": "y"},
}


@pytest.mark.parametrize("integ", ["simple", "hierarchical"])
@pytest.mark.parametrize("name", list(DEFORM))
@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 1, 5), (4, 4, 4), (5, 3, 4), (17, 16, 33)])
def test_voxel_root_fp64(ctx, monkeypatch, shape, name, integ):
    rho = np.random.default_rng(7).random(shape, dtype=np.float32)
    rho[shape[0] // 2:, :, : shape[2] // 2] = 0.0
    res, ds = 27, 0.06
    sc = xrp_scene(None, DEFORM[name], voxels=rho)
    kw = dict(integrator=integ, precision="fp64")
    # the linear copy alone is made resident first
    monkeypatch.setenv("XRP_VOXEL_LAYOUT", "linear")
    X.render(ctx, sc, ANGLES, 4, 0.5, integrator="simple", precision="guarded")
    import torch
    out = torch.zeros((2, res, res), dtype=torch.float32, device="cuda")
    sl = X.render_device_noalloc(ctx, sc, ANGLES, res, ds, out.data_ptr(), **kw)
    linear = out.cpu().numpy()
    img, st = X.render(ctx, sc, ANGLES, res, ds, **kw)
    sc.close()
    assert np.array_equal(img, linear)
    assert st["samples"] == sl["samples"] and st["fine_samples"] == sl["fine_samples"]
    osc = oracle_scene(None, DEFORM[name], rho)
    ref = oracle_render(osc, ANGLES, res, ds, integrator=integ)
    assert float(np.abs(img.astype(np.float64) - ref).max()) <= 1e-5
