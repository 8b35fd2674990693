"""The backward of 64-wide networks (weight gradients as split-bf16 products through transposing LDS reads) where its
split of the work can go wrong: one tile, a partial tile, one phase only, several rounds with a ragged last one, widths
that leave padded features, a 64-wide network beside a narrow one, one hidden layer's or several layers' blocks.

Reference: the same records in float64 with torch autograd.  Bars as in test_gpu_mfma.py (1e-5 on the loss, 1e-4 on
the gradient, 2-norm): float32 rounding of the forward pass dominates both.  The recomputing variant runs
the same groups and sums, hence gives the same bits.
"""
import ctypes

import numpy as np
import pytest


def records(rows, per_row, plus_share, seed):
    """Random rows of random offsets around the points of a small grid."""
    from jax_dips.records import DeviceGrid, DeviceRecords, pack_dense

    rng = np.random.default_rng(seed)
    n = int(np.ceil(rows ** (1 / 3))) + 1
    axes = [np.linspace(-1, 1, n, dtype=np.float32)] * 3
    W = np.zeros((rows, 250))
    for r in range(rows):
        q = rng.choice(125, per_row, replace=False)
        W[r, 2 * q + (rng.random(per_row) < plus_share)] = rng.normal(size=per_row)
    packed = pack_dense(W, rng.normal(size=rows), rows)
    return DeviceGrid(*axes), DeviceRecords(packed, np.full(3, 0.037, np.float32))


def reference(grid, rec, dims, theta):
    import torch

    th = theta.double().requires_grad_(True)
    ptr = rec.row_ptr.long()
    row = torch.repeat_interleave(torch.arange(rec.nrows, device="cuda"), ptr[1:] - ptr[:-1])
    code = rec.ent_code[:rec.nnz].long()
    k = code & 127
    o = torch.stack([k % 5 - 2, k // 5 % 5 - 2, k // 25 - 2], 1).float()
    x = (grid.points()[rec.row_point.long()[row]] + o * torch.as_tensor(rec.h, device="cuda")).double()
    Lm, Hm, Lp, Hp = dims
    u, off = [], 0
    for L, H in ((Lp, Hp), (Lm, Hm)):
        a = x
        for i, (m, n) in enumerate([(3, H)] + [(H, H)] * (L - 1) + [(H, 1)]):
            a = a @ th[off:off + m * n].view(m, n) + th[off + m * n:off + m * n + n]
            off += m * n + n
            if i < L:
                a = torch.tanh(a)
        u.append(a[:, 0])
    v = torch.where((code & 128) != 0, u[0], u[1]) * rec.ent_w[:rec.nnz].double()
    r = rec.row_c.double().index_add(0, row, v)
    loss = 0.5 * (r * r).sum() / rec.nrows
    (g,) = torch.autograd.grad(loss, th)
    return loss.item(), g


CASES = [((3, 64, 3, 64), 1, 1, 1.0), ((3, 64, 3, 64), 2, 7, 0.0), ((3, 64, 3, 64), 5, 13, 0.5),
         ((3, 64, 3, 64), 3000, 9, 0.3), ((3, 64, 3, 64), 6000, 13, 0.97), ((3, 50, 3, 61), 3000, 9, 0.5),
         ((1, 7, 3, 64), 4000, 11, 0.5), ((3, 64, 3, 64), 5000, 9, 1.0)]


@pytest.mark.gpu
@pytest.mark.parametrize("dims,rows,per_row,share", CASES)
def test_split_backward(dims, rows, per_row, share):
    import torch

    from jax_dips import _native as N
    from jax_dips.records import Engine

    grid, rec = records(rows, per_row, share, rows + per_row)
    g = torch.Generator().manual_seed(rows)
    Lm, Hm, Lp, Hp = dims
    parts = []
    for L, H in ((Lp, Hp), (Lm, Hm)):
        for a, b in [(3, H)] + [(H, H)] * (L - 1) + [(H, 1)]:
            parts += [torch.randn(a * b, generator=g) / a ** 0.5, 0.1 * torch.randn(b, generator=g)]
    theta = torch.cat(parts)
    eng = Engine(dims, theta.numpy(), {}, max_rows=rows, max_steps=4)
    ref_loss, ref_g = reference(grid, rec, dims, theta.cuda())

    mb = eng.mfma_workspace(rec, grid, grouped=False)
    L = N.lib()
    outs = []
    full = int(L.dips_mfma_workspace(ctypes.byref(eng.net), rows, mb["max_nnz"]))
    # the same step with and without room for the stored activations
    act_f4 = max((Lm - 1) * -(-Hm // 16), (Lp - 1) * -(-Hp // 16))
    small = full - (mb["max_nnz"] // 16 + 2) * act_f4 * 256 - 64
    for floats in (full, small):
        grad = torch.empty(eng.P, dtype=torch.float32, device="cuda")
        loss = torch.empty(1, dtype=torch.float64, device="cuda")
        N.check(L.dips_mfma_loss_grad(ctypes.byref(grid.c), ctypes.byref(rec.c), ctypes.byref(mb["batches"][0]),
                                      ctypes.byref(eng.net), ctypes.c_float(1.0 / rows), N.ptr(eng.params), N.ptr(grad),
                                      N.ptr(loss), N.ptr(eng._mwork), floats, N.ptr(eng._mdwork),
                                      int(eng._mdwork.numel()), N.current_stream()), "dips_mfma_loss_grad")
        torch.cuda.synchronize()
        outs.append((float(loss), grad))
    assert abs(outs[0][0] - ref_loss) <= 1e-5 * abs(ref_loss)
    assert float((outs[0][1].double() - ref_g).norm()) <= 1e-4 * float(ref_g.norm())
    assert outs[0][0] == outs[1][0] and torch.equal(outs[0][1], outs[1][1])
    # a network without entries has no gradient
    PP = 4 * Hp + (Lp - 1) * (Hp * Hp + Hp) + Hp + 1
    if share == 0.0:
        assert not bool(outs[0][1][:PP].any())
    if share == 1.0:
        assert not bool(outs[0][1][PP:].any())
