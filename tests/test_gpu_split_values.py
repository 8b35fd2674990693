"""Values of the split-bf16 weight gradients of 64-wide networks where the split itself decides them."""
import ctypes

import numpy as np
import pytest

DIMS = (3, 64, 3, 64)
P1 = 4 * 64 + 2 * (64 * 64 + 64) + 65  # parameters of one network


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
