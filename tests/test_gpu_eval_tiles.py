"""dips_eval on the MFMA path at the edges of its tiles: point counts around a tile, a workgroup's tiles and one
round of the grid, all points in one phase, both phases inside a tile, each combination of outputs.

Reference: the same networks in float64 with torch autograd.  Tolerance: a hidden activation is within 5e-7 of
its float64 value (4e-7 for the hardware tanh, the rest the rounding of a 64-term product), which three layers
of unit gain accumulate to 1.5e-6 in u (of order 0.3 here): 5e-6 relative in the 2-norm; the gradient passes back through the
same layers: 1e-5.
"""
import ctypes

import numpy as np
import pytest


def nets64(theta, dims, x):
    import torch

    Lm, Hm, Lp, Hp = dims
    out, o = [], 0
    for L, H in ((Lp, Hp), (Lm, Hm)):
        a = x
        for i, (m, n) in enumerate([(3, H)] + [(H, H)] * (L - 1) + [(H, 1)]):
            W, b = theta[o:o + m * n].view(m, n), theta[o + m * n:o + m * n + n]
            o += m * n + n
            a = a @ W + b
            if i < L:
                a = torch.tanh(a)
        out.append(a[:, 0])
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(3, 64, 3, 64), (3, 50, 3, 64), (3, 32, 3, 32), (2, 12, 2, 16), (1, 12, 3, 64)])
@pytest.mark.parametrize("m,mix", [(1, "plus"), (15, "minus"), (16, "mixed"), (17, "mixed"), (12 * 16 + 1, "blocks"),
                                   (256 * 12 * 16 + 5, "blocks"), (100003, "mixed"), (4097, "plus")])
def test_eval_tiles(dims, m, mix):
    import torch

    from jax_dips import _native as N

    g = torch.Generator().manual_seed(m + sum(dims))
    Lm, Hm, Lp, Hp = dims
    parts = []
    for L, H in ((Lp, Hp), (Lm, Hm)):
        for a, b in [(3, H)] + [(H, H)] * (L - 1) + [(H, 1)]:
            parts += [torch.randn(a * b, generator=g) / a ** 0.5, 0.1 * torch.randn(b, generator=g)]
    theta = torch.cat(parts).cuda()
    pts = (2 * torch.rand(m, 3, generator=g) - 1).cuda()
    nrm = torch.randn(m, 3, generator=g).cuda()
    i = torch.arange(m)
    phase = {"plus": i >= 0, "minus": i < 0, "mixed": torch.rand(m, generator=g) < 0.5, "blocks": i // 40 % 3 == 0}[mix]
    ph = phase.to(torch.uint8).cuda()
    net = N.Net(*dims, 0, 0, 0.0, 0)
    assert N.lib().dips_mfma_supported(ctypes.byref(net)) and not N.lib().dips_net_supported(ctypes.byref(net))

    def run(want_grad, want_n):
        u, gr, gn = (torch.full(s, 7.0, device="cuda") for s in ((m,), (m, 3), (m,)))
        N.check(N.lib().dips_eval(ctypes.byref(net), N.ptr(theta), N.ptr(pts), N.ptr(ph), N.ptr(nrm) if want_n else None,
                                  m, N.ptr(u), N.ptr(gr) if want_grad else None, N.ptr(gn) if want_n else None,
                                  N.current_stream()), "dips_eval")
        torch.cuda.synchronize()
        return u, gr, gn

    u, gr, gn = run(True, True)
    x = pts.double().requires_grad_(True)
    up, um = nets64(theta.double(), dims, x)
    ref = torch.where(phase.cuda(), up, um)
    (gref,) = torch.autograd.grad(ref.sum(), x)
    nref = (gref * nrm.double()).sum(1)

    def rel(a, b):
        return float((a.double() - b).norm() / b.norm())

    assert rel(u, ref.detach()) <= 5e-6
    assert rel(gr, gref) <= 1e-5
    assert float((gn.double() - nref).norm()) <= 1e-5 * float((gref.norm(dim=1) * nrm.double().norm(dim=1)).norm())
    u1, gr1, gn1 = run(True, False)
    assert torch.equal(gr1, gr) and torch.equal(u1, u) and bool((gn1 == 7.0).all())
    u2, gr2, gn2 = run(False, False)
    assert rel(u2, ref.detach()) <= 5e-6 and bool((gr2 == 7.0).all()) and bool((gn2 == 7.0).all())
    u3, gr3, gn3 = run(False, True)
    assert torch.equal(gn3, gn) and bool((gr3 == 7.0).all())


@pytest.mark.gpu
def test_eval_extreme_weights():
    """An infinite or very large hidden weight saturates its unit, a NaN one makes u NaN (as in float64)."""
    import torch

    from jax_dips import _native as N

    dims, m = (3, 64, 3, 64), 100
    g = torch.Generator().manual_seed(1)
    P = 4 * 64 + 2 * (64 * 64 + 64) + 65
    theta = (0.2 * torch.randn(2 * P, generator=g)).cuda()
    theta[256 + 5], theta[256 + 64 * 7 + 9], theta[256 + 64 * 9 + 11] = float("inf"), -3.4e38, 1e38
    pts = (2 * torch.rand(m, 3, generator=g) - 1).cuda()
    ph = torch.ones(m, dtype=torch.uint8, device="cuda")
    net = N.Net(*dims, 0, 0, 0.0, 0)
    u = torch.empty(m, device="cuda")

    def run(th):
        N.check(N.lib().dips_eval(ctypes.byref(net), N.ptr(th), N.ptr(pts), N.ptr(ph), None, m, N.ptr(u), None, None,
                                  N.current_stream()), "dips_eval")
        return u.double()

    ref, _ = nets64(theta.double(), dims, pts.double())
    assert bool(torch.isfinite(ref).all())
    assert float((run(theta) - ref).norm() / ref.norm()) <= 5e-6
    theta[256 + 5] = float("nan")
    assert bool(torch.isnan(run(theta)).all())
