"""Results copied to the caller's pageable memory (api.cpp copy_to_host): sizes
about the least that passes through the pinned slots, ragged last chunks, and
destinations that are pinned or not aligned, against the device's own copy."""
import ctypes

import numpy as np
import pytest
import torch

import xray_projection_render_amd as X
from xray_projection_render_amd import _lib
from helpers import xrp_scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("views,res", [(32, 512), (31, 511), (33, 509), (64, 363), (3, 2048)])
@pytest.mark.parametrize("where", ["numpy", "odd", "pinned"])
def test_render_to_host(ctx, views, res, where):
    sc = xrp_scene({"type": "sphere", "center": [0.1, 0.0, -0.1], "radius": 0.5, "rho": 1.0})
    angles = [(360.0 * k / views, 90.0) for k in range(views)]
    dev = torch.zeros((views, res, res), dtype=torch.float32, device="cuda")
    kw = dict(integrator="simple")
    X.render_device(ctx, sc, angles, res, 0.05, dev.data_ptr(), **kw)
    n = views * res * res
    if where == "pinned":
        keep = torch.empty(n, dtype=torch.float32, pin_memory=True)
        out = keep.numpy()
    elif where == "odd":
        out = np.zeros(n + 1, dtype=np.float32)[1:]
    else:
        out = np.zeros(n, dtype=np.float32)
    p, st = _lib.make_params(res, 0.05, **kw), _lib.RenderStats()
    _lib.check(_lib.lib().xrp_render(ctx.ptr, sc.ptr, ctypes.byref(p), _lib._views(angles), views,
                                     ctypes.c_void_p(out.ctypes.data), ctypes.byref(st)))
    sc.close()
    assert np.array_equal(out.reshape(views, res, res), dev.cpu().numpy())
