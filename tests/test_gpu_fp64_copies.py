"""FP64 renders of a voxel root that go without the quad copy."""
import numpy as np
import pytest
import torch

import xray_projection_render_amd as X
from helpers import xrp_scene

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 75.0), (130.0, 100.0)]
HIER = dict(integrator="hierarchical")


def _grid(n):
    return np.random.default_rng(4).random((n, n, n), dtype=np.float32)


def test_fallback_leaves_no_error_text(monkeypatch):
    """A render without allocation that finds no quad copy reads the linear
    one and succeeds: the thread's last error text stays what it was."""
    out = torch.zeros((2, 24, 24), dtype=torch.float32, device="cuda")
    with X.Context(0) as ctx:
        sc = xrp_scene(None, None, _grid(12))
        monkeypatch.setenv("XRP_VOXEL_LAYOUT", "linear")
        X.render(ctx, sc, ANGLES, 24, 0.05, integrator="simple")  # the linear copy alone
        monkeypatch.delenv("XRP_VOXEL_LAYOUT")
        with pytest.raises(X.XrpError):
            X.render(ctx, sc, ANGLES, 24, -0.05)
        before = X.lib().xrp_last_error()
        X.render_device_noalloc(ctx, sc, ANGLES, 24, 0.05, out.data_ptr(), **HIER)
        assert X.lib().xrp_last_error() == before
        want, _ = X.render(ctx, sc, ANGLES, 24, 0.05, **HIER)  # from the quads
        sc.close()
    assert np.array_equal(out.cpu().numpy(), want)
