"""Values of the split-bf16 weight gradients of 64-wide networks where the split itself decides them."""
import ctypes

import numpy as np
import pytest

DIMS = (3, 64, 3, 64)
P1 = 4 * 64 + 2 * (64 * 64 + 64) + 65  # parameters of one network
LAYERS = {"W0": 0, "b0": 192, "W1": 256, "b1": 4352, "W2": 4416, "b2": 8512, "wo": 8576}


def gradient(points, weight, const, plus, theta):
    """Gradient of a batch with one entry (weight, phase) per point, at the point; both workspace sizes."""
    import torch

    from jax_dips import _native as N
    from jax_dips.records import DeviceGrid, DeviceRecords, Engine, pack_dense

    n = len(points)
    W = np.zeros((n, 250))
    W[np.arange(n), 2 * 62 + plus.astype(int)] = weight
    grid, rec = DeviceGrid.from_points(points), DeviceRecords(pack_dense(W, const, n), np.full(3, 0.1, np.float32))
    eng = Engine(DIMS, theta, {}, max_rows=n, max_steps=4)
    mb = eng.mfma_workspace(rec, grid, grouped=False)
    L = N.lib()
    full = int(L.dips_mfma_workspace(ctypes.byref(eng.net), n, mb["max_nnz"]))
    out = []
    for floats in (full, full - (mb["max_nnz"] // 16 + 2) * 8 * 256 - 64):  # activations stored, recomputed
        g = torch.empty(eng.P, dtype=torch.float32, device="cuda")
        loss = torch.empty(1, dtype=torch.float64, device="cuda")
        N.check(L.dips_mfma_loss_grad(ctypes.byref(grid.c), ctypes.byref(rec.c), ctypes.byref(mb["batches"][0]),
                                      ctypes.byref(eng.net), ctypes.c_float(1.0), N.ptr(eng.params), N.ptr(g),
                                      N.ptr(loss), N.ptr(eng._mwork), floats, N.ptr(eng._mdwork),
                                      int(eng._mdwork.numel()), N.current_stream()), "dips_mfma_loss_grad")
        out.append(g.cpu().numpy())
    assert np.array_equal(out[0], out[1], equal_nan=True)
    return out[0]


@pytest.mark.gpu
def test_products_have_no_common_sign():
    """With every point of a batch at one x and y, dW0[x] = x db0 exactly.  The terms that a product of two split operands
    drops must not add up: with both cut off by truncation, parts have their operand's sign and dW0 comes out 3.8e-8 short
    (on average x1 / x = 2.7e-3 and x2 / x = 7e-6, for x and for the deltas).  Without a common sign an x leaves 2e-8
    of either sign; 16 of them on two axes 3.5e-9, and the float32 rounding of the 4096 sums less: 1.5e-8."""
    rng = np.random.default_rng(3)
    n, short = 1024, []
    theta = 0.1 * rng.normal(size=2 * P1).astype(np.float32)
    for _ in range(16):
        xy = rng.uniform(0.5, 1.0, 2).astype(np.float32)
        pts = np.stack([np.full(n, xy[0]), np.full(n, xy[1]), 1e-3 * rng.random(n)], 1).astype(np.float32)
        g = gradient(pts, 1 + rng.random(n), 5 + 5 * rng.random(n), np.arange(n) % 2 == 0, theta).astype(np.float64)
        short += [g[o + 64 * k:o + 64 * k + 64] / (g[o + 192:o + 256] * float(xy[k])) - 1 for o in (0, P1) for k in (0, 1)]
    assert np.abs(short).max() <= 1e-6
    assert abs(np.mean(short)) <= 1.5e-8, np.mean(short)


@pytest.mark.gpu
@pytest.mark.parametrize("layer,delta", [(2, np.inf), (1, 1.5e38), (0, 6e37)])
def test_infinite_deltas(layer, delta):
    """One row's deltas overflow float32 at a layer (delta: at the last one; a layer multiplies them by 3.7 here, the
    factor of the packed weights among it): that layer's gradients of the row's network are infinite with the sign of their
    products, as float32 products give them; the other network's stay finite."""
    rng = np.random.default_rng(layer)
    n, hot = 301, 147
    pts = (0.2 + 0.6 * rng.random((n, 3))).astype(np.float32)
    theta = np.zeros(2 * P1, np.float32)
    for o in (0, P1):
        theta[o:o + 192] = 0.4 * rng.uniform(-1, 1, 192)
        theta[o + 256:o + 8512] = 0.02
        for name in ("b1", "b2"):
            theta[o + LAYERS[name]:o + LAYERS[name] + 64] = 0.1
        theta[o + 8576:o + 8640] = 1.0
    weight, const = 1 + rng.random(n), rng.normal(size=n)
    a = pts[hot].astype(np.float64) @ theta[:192].reshape(3, 64).astype(np.float64)
    acts = [np.tanh(a)]
    for name in ("1", "2"):
        acts.append(np.tanh(acts[-1] @ np.full((64, 64), float(np.float32(0.02))) + 0.1))
    w = 1e20
    u = acts[2].sum()
    weight[hot] = w
    const[hot] = 1e20 if np.isinf(delta) else delta / (w * (1 - acts[2][0] ** 2)) - w * u
    plus = np.arange(n) % 2 == 1
    g = gradient(pts, weight, const, plus, theta)
    below = pts[hot] if layer == 0 else acts[layer - 1]
    blk = g[LAYERS["W%d" % layer]:][:below.size * 64].reshape(-1, 64)
    assert np.array_equal(blk, np.broadcast_to(np.copysign(np.inf, below)[:, None], blk.shape))
    assert np.all(g[LAYERS["b%d" % layer]:][:64] == np.inf)
    assert np.all(np.isfinite(g[P1:])) and np.any(g[P1:])
