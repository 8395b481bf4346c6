"""The surrogate's gradients by the two ways of adding to the tables: by slices
(a workgroup each, or shared out over parts of the samples), and, for tables of
more slices than that pays for (2^22 entries and up), by adds in global memory.
XRP_SUR_SLICES, read per batch, takes small tables the second way."""
import numpy as np
import pytest

import xray_projection_render_amd as X
from test_gpu_surrogate_train import S, TOL, _loss_and_grads, _net

pytestmark = pytest.mark.gpu


def _samples(rng, n):
    u = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    return u, (rng.uniform(0, 1, n) > 0.6).astype(np.float32)


@pytest.mark.parametrize("log2_table,n", [(4, 500), (13, 1), (13, 17), (14, 1000),
                                          (13, (1 << 17) + 4099)])  # past a chunk
def test_global_adds_give_the_sliced_gradients(ctx, monkeypatch, log2_table, n):
    """The same terms in another order.  An entry of m terms is off by sqrt(m)
    2^-24 of their sizes' sum, and that sum is at most about sqrt(m) times the
    result (signs at random): m 2^-24, with m = 8 n / 9^3 entries of the coarsest
    level 9e-5 at most; the MLP's sums are made the same way in both."""
    sur, _, rng = _net(ctx, log2_table, 8, 64)
    u, t = _samples(rng, n)
    sliced, la = sur.gradients(u, t)
    monkeypatch.setenv("XRP_SUR_SLICES", "0")
    direct, lb = sur.gradients(u, t)
    monkeypatch.delenv("XRP_SUR_SLICES")
    sur.close()
    a, b = (X.split_surrogate_params(g.astype(np.float64), log2_table) for g in (sliced, direct))
    rel = np.linalg.norm(a["tables"] - b["tables"]) / np.linalg.norm(a["tables"])
    print(f"2^{log2_table} entries, {n} samples: rel {rel:.1e}", flush=True)
    assert rel <= 1e-3
    for name in ("W1", "b1", "W2", "b2", "w3", "b3"):
        assert np.array_equal(a[name], b[name]), name
    assert abs(la - lb) <= 1e-9 * la


@pytest.mark.parametrize("slices", [None, "0"])
def test_tables_of_many_slices(ctx, monkeypatch, slices):
    """2^18 entries: 32 slices a level, one workgroup each."""
    if slices:
        monkeypatch.setenv("XRP_SUR_SLICES", slices)
    sur, p, rng = _net(ctx, 18, 16, 512)
    u, t = _samples(rng, 1000)
    g, loss = sur.gradients(u, t)
    sur.close()
    cfg = S.Config(log2_table=18, n_min=16, n_max=512)
    loss_ref, ref = _loss_and_grads(u.astype(np.float64), t.astype(np.float64), p, cfg)
    assert abs(loss - loss_ref) <= 1e-4 * loss_ref
    got = X.split_surrogate_params(g.astype(np.float64), 18)
    for name in ("tables", "W1", "b1", "W2", "b2", "w3", "b3"):
        a, b = np.asarray(got[name]), np.asarray(ref[name])
        assert np.linalg.norm(a - b) <= TOL * max(np.linalg.norm(b), 1e-30), name
    assert (np.asarray(got["tables"])[ref["tables"] == 0.0] == 0.0).all()
