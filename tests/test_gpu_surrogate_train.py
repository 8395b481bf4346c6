"""The surrogate's gradients at the edges of their kernels: tables of less than
a slice, of one and of many, levels shared out over parts of the samples, and
sample counts about a group, a launch and a chunk, against the restatement
(oracle/surrogate_ref.py) with the kernels' BF16 roundings in it, and against
their own sums over parts.

With the same roundings, what is left is FP32 against FP64: about 1e-6 of an
operand, which moves 3e-4 of the roundings by 2^-8, hence 7e-5 of a gradient,
and up to 30 times as much of one whose samples mostly cancel."""
import math
import os
import sys

import numpy as np
import pytest

import xray_projection_render_amd as X
from xray_projection_render_amd import workloads as W
from helpers import ROOT, xrp_scene

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import surrogate_ref as S  # noqa: E402

pytestmark = pytest.mark.gpu

TOL = 1e-2


def _bf16(a):
    b = np.asarray(a, dtype=np.float32).view(np.uint32)
    b = (b + 0x7FFF + ((b >> 16) & 1)) & np.uint32(0xFFFF0000)
    return b.view(np.float32).astype(np.float64)


def _loss_and_grads(u, t, p, cfg):
    x, cache = S.encode(u, p["tables"].astype(np.float32).astype(np.float64), cfg)
    x, w1, w2 = _bf16(x), _bf16(p["W1"]), _bf16(p["W2"])
    z1 = x @ w1 + p["b1"]
    h1 = _bf16(np.maximum(z1, 0.0))
    z2 = h1 @ w2 + p["b2"]
    h2 = np.maximum(z2, 0.0)
    y = 1.0 / (1.0 + np.exp(-(h2 @ p["w3"] + p["b3"])))
    dz = 2.0 * (y - t) / len(u) * y * (1.0 - y)
    d2 = np.outer(dz, p["w3"]) * (z2 > 0)
    d1 = (_bf16(d2) @ w2.T) * (z1 > 0)
    dx = _bf16(d1) @ w1.T
    g = {"b3": dz.sum(), "w3": h2.T @ dz, "b2": d2.sum(0), "W2": h1.T @ _bf16(d2),
         "b1": d1.sum(0), "W1": x.T @ _bf16(d1), "tables": np.zeros_like(p["tables"])}
    for l, (idx, wts) in enumerate(cache):
        for f in range(2):
            np.add.at(g["tables"][l, :, f], idx, wts * dx[:, 2 * l + f][:, None])
    return float(np.mean((y - t) ** 2)), g


def _net(ctx, log2_table, n_min, n_max):
    w = W.gyroid_lattice(resolution=16, n_views=1)
    sur = X.Surrogate(ctx, xrp_scene(w.obj, None), log2_table=log2_table, n_min=n_min,
                      n_max=n_max)
    rng = np.random.default_rng(log2_table)
    p = {
        "tables": rng.uniform(-0.5, 0.5, (16, 1 << log2_table, 2)),
        "W1": rng.normal(0, 1 / math.sqrt(32), (32, 64)),
        "b1": rng.normal(0, 0.1, 64),
        "W2": rng.normal(0, 1 / math.sqrt(64), (64, 64)),
        "b2": rng.normal(0, 0.1, 64),
        "w3": rng.normal(0, 1 / math.sqrt(64), 64),
        "b3": np.float64(0.2),
    }
    sur.set_params(X.join_surrogate_params(p))
    return sur, p, rng


@pytest.mark.parametrize("log2_table,n_min,n_max,n", [
    (4, 2, 16, 500),       # 16 entries: every add on the same few
    (12, 4, 64, 1),        # one sample
    (13, 4, 128, 17),      # one slice of exactly the table; a group and one more
    (14, 16, 256, 1000),
    (16, 16, 512, 16385),  # 8 slices; more than one group a wave
])
def test_gradients_at_the_edges(ctx, log2_table, n_min, n_max, n):
    sur, p, rng = _net(ctx, log2_table, n_min, n_max)
    u = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    u[0] = [1.0, 0.0, 1.0]
    t = (rng.uniform(0, 1, n) > 0.6).astype(np.float32)
    g, loss = sur.gradients(u, t)
    sur.close()
    cfg = S.Config(log2_table=log2_table, n_min=n_min, n_max=n_max)
    loss_ref, g_ref = _loss_and_grads(u.astype(np.float64), t.astype(np.float64), p, cfg)
    assert abs(loss - loss_ref) <= 1e-4 * loss_ref
    gg = X.split_surrogate_params(g.astype(np.float64), log2_table)
    for name in ("tables", "W1", "b1", "W2", "b2", "w3", "b3"):
        a, b = np.asarray(gg[name]), np.asarray(g_ref[name])
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        print(f"{name}: rel {rel:.3e}", flush=True)
        assert rel < TOL, name
    # an entry that no sample's corner reaches has no gradient
    assert (np.asarray(gg["tables"])[g_ref["tables"] == 0.0] == 0.0).all()


def test_gradients_over_chunks(ctx):
    """More samples than one launch takes: n times the mean's gradient is the sum
    over two parts, to the FP32 rounding of sums of up to n terms."""
    sur, _, rng = _net(ctx, 13, 8, 64)
    n, m = (1 << 17) + 4099, 70001
    u = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    t = (rng.uniform(0, 1, n) > 0.6).astype(np.float32)
    whole, lw = sur.gradients(u, t)
    a, la = sur.gradients(u[:m], t[:m])
    b, lb = sur.gradients(u[m:], t[m:])
    sur.close()
    parts = (m * a.astype(np.float64) + (n - m) * b.astype(np.float64)) / n
    rel = np.linalg.norm(whole - parts) / np.linalg.norm(parts)
    print(f"rel {rel:.2e}", flush=True)
    # rounding of n terms in a random walk, sqrt(n) 2^-24, and BF16 values of the
    # output gradients scaled by 1 / n (2^-9 each, as often up as down)
    assert rel <= 2e-3
    assert abs(lw - (m * la + (n - m) * lb) / n) <= 1e-6 * lw
