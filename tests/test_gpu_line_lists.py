"""Device memory of the interval march's two passes: the list of rays to march
again, and none of the lists that only the other marches fill."""
import pytest
import torch

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import xrp_scene

pytestmark = pytest.mark.gpu


def test_two_passes_allocate_the_redo_list_alone():
    views, res = 4, 1024
    w = W.lattice(resolution=res, n_views=views, ds=0.01)
    out = torch.zeros((views, res, res), dtype=torch.float32, device="cuda")
    with X.Context(0) as ctx:
        sc = xrp_scene(w.obj, w.deformation)
        X.render_device(ctx, sc, w.angles[:1], 64, w.ds, out.data_ptr())  # one pass: no list
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        st = X.render_device(ctx, sc, w.angles, res, w.ds, out.data_ptr())
        torch.cuda.synchronize()
        grown = before - torch.cuda.mem_get_info()[0]
        sc.close()
    rays = views * res * res
    print(f"{rays} rays: {grown >> 20} MiB", flush=True)
    assert st["two_pass"] == 1
    # 4 bytes a ray, up to 2^22 of them; 4 MiB for the allocator's granularity
    assert grown <= 4 * rays + (4 << 20)
