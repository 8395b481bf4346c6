"""The quad copy of FP64 renders of a voxel root: what builds it, and the renders
that go without."""
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


def _used():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


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


def test_audit_keeps_the_grid_alone(monkeypatch):
    """An audited render, made to check others once, keeps no copy beside the
    grid; nor does any FP64 render under XRP_FP64_QUADS=0.  Both give the bits of
    the renders that read the quads."""
    n = 256
    grid = _grid(n)
    with X.Context(0) as ctx:
        small = xrp_scene(None, None, _grid(8))
        X.render(ctx, small, ANGLES, 24, 0.05, **HIER)  # the context's own buffers
        small.close()
        sc = xrp_scene(None, None, grid)
        start = _used()
        audit, _ = X.render(ctx, sc, ANGLES, 24, 0.05, audit=True, **HIER)
        after_audit = _used() - start
        monkeypatch.setenv("XRP_FP64_QUADS", "0")
        linear, _ = X.render(ctx, sc, ANGLES, 24, 0.05, **HIER)
        after_linear = _used() - start
        monkeypatch.delenv("XRP_FP64_QUADS")
        quads, _ = X.render(ctx, sc, ANGLES, 24, 0.05, **HIER)
        after_quads = _used() - start
        sc.close()
    print(f"grid {grid.nbytes >> 20} MiB: {after_audit >> 20}, {after_linear >> 20}, "
          f"{after_quads >> 20} MiB", flush=True)
    assert np.array_equal(audit, quads) and np.array_equal(linear, quads)
    assert after_audit < 2 * grid.nbytes and after_linear < 2 * grid.nbytes
