"""Volume uploads of one context do not hold up the others: a call that copies a
large volume over leaves the process-wide scene registry free meanwhile."""
import threading
import time

import numpy as np
import pytest

import xray_projection_render_amd as X
from helpers import xrp_scene

pytestmark = pytest.mark.gpu


def test_registry_is_free_during_a_volume_upload(ctx):
    """Half a gigabyte a call; meanwhile another thread creates and destroys
    scenes, which registers nothing on a device and takes that lock alone.  With
    the lock held over the upload nearly every one waited for a large part of a
    call; free, each takes far less."""
    vol = np.zeros((512, 512, 512), dtype=np.float32)
    cams = [X.camera_from_angles(20.0, 90.0, 4.0) + (40.0, 4.0)]
    sphere = {"type": "sphere", "center": [0.0, 0.0, 0.0], "radius": 0.3, "rho": 1.0}
    calls, done = [], threading.Event()

    def uploads():
        for _ in range(12):
            t = time.perf_counter()
            X.render_volume_projections(ctx, vol, cams, 8, 0.5)
            calls.append(time.perf_counter() - t)
        done.set()

    X.render_volume_projections(ctx, vol, cams, 8, 0.5)  # buffers and copies exist
    th = threading.Thread(target=uploads)
    th.start()
    waits = []
    while not done.is_set():
        sc = xrp_scene(sphere)
        t = time.perf_counter()
        sc.close()
        waits.append(time.perf_counter() - t)
        time.sleep(0.0005)
    th.join()
    X.render_volume_projections(ctx, vol[:4, :4, :4].copy(), cams, 8, 0.5)  # the large one goes
    call, wait = float(np.median(calls)), sorted(waits)
    print(f"call {1e3 * call:.1f} ms, {len(waits)} destroys: median "
          f"{1e3 * wait[len(wait) // 2]:.3f} ms, worst {1e3 * wait[-1]:.1f} ms", flush=True)
    assert wait[len(wait) // 2] < 0.1 * call
