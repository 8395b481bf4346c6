"""The guard band of the gyroid march (api.cpp gyroid_plan) covers every rounding
of its FP32 level: gyroids whose centre is far from the box (the lattice is
periodic, so any centre is legal) and unit cells away from the origin, audited
sample by sample in FP64.

The centre's coordinates are half an FP32 ulp off an FP32 number, all to the
same side, so that its own rounding is as large as it can be; positions less
such a centre round by as much again.  The general march (XRP_GYROID=0), whose
band counts both, gives the same bits."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import xrp_scene

pytestmark = pytest.mark.gpu

ANGLES = [(20.0, 90.0), (0.0, 90.0), (133.0, 61.0)]
HALF_ULP = 0.999 * 2.0 ** -14  # of numbers from 1024 to 2048
# centre, offset of the unit cell in cells, offset of the box
PLACES = [([1024.0 + HALF_ULP] * 3, [0.0] * 3, [0.0] * 3),
          ([-1024.0 - HALF_ULP] * 3, [0.0] * 3, [0.0] * 3),
          ([1024.0 + HALF_ULP, -5.3, 64.0 + 0.999 * 2.0 ** -18], [7.0, -11.0, 0.5], [0.0] * 3),
          ([0.01, 0.02, -0.03], [40.0, 0.0, -25.0], [0.2, -0.3, 0.1])]


def _object(place, cells=6):
    centre, off, shift = place
    obj = W.gyroid_lattice(resolution=16, n_views=1, cells=cells).obj
    obj["uc"]["objects"]["objects"][0]["center"] = centre
    for a, k in zip("xyz", range(3)):
        for end in ("min", "max"):
            obj["uc"][a + end] += off[k] / cells
            obj[a + end] += shift[k]
    return obj


@pytest.mark.parametrize("integ", ["simple", "hierarchical"])
@pytest.mark.parametrize("shear", [False, True])
@pytest.mark.parametrize("place", range(len(PLACES)))
def test_band_covers_far_centres(ctx, monkeypatch, place, shear, integ):
    sc = xrp_scene(_object(PLACES[place]), W.TANH_SHEAR if shear else None)
    ds = 0.002 if integ == "simple" else 0.01
    kw = dict(integrator=integ, precision="guarded")
    out = {}
    for on in ("1", "0"):
        monkeypatch.setenv("XRP_GYROID", on)
        out[on], _ = X.render(ctx, sc, ANGLES, 96, ds, **kw)
    monkeypatch.delenv("XRP_GYROID")
    _, st = X.render(ctx, sc, ANGLES, 96, ds, audit=True, **kw)
    sc.close()
    print(f"place {place} {integ}: audit mismatches {st['audit_mismatch']}, differing pixels "
          f"{int(np.count_nonzero(out['1'] != out['0']))}", flush=True)
    assert st["audit_mismatch"] == 0
    assert np.array_equal(out["1"], out["0"])
