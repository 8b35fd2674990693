"""The grid operator's rows and the solver's sizes at the edges of their work split: rows of every length around
a round of entries, partial workgroups and groups of workgroups, box rows reading the ghost layer; solves whose
inner products need one workgroup, few, and more than the float64 workspace holds beside each other.

Tolerances: a row of L entries is a float32 chain of L fused multiply-adds, |error| <= (L + 1) 2^-24 sum |w u|
(the ghost values add two roundings of their terms, covered by 4x); a solve stops at a relative residual of
1e-6 of the recurrence, whose float32 iterate drifts from the true residual by a few times that (10x).
"""
import ctypes

import numpy as np
import pytest

from jax_dips import problems


def ghost(u, idx, shape):
    """Linear extrapolation one node beyond the box, per axis (numpy, float64)."""
    terms = [(1.0, ())]
    for a, n in zip(idx, shape):
        if a < 0:
            rule = [(2.0, 0), (-1.0, 1)]
        elif a >= n:
            rule = [(2.0, n - 1), (-1.0, n - 2)]
        else:
            rule = [(1.0, a)]
        terms = [(w * r, t + (i,)) for w, t in terms for r, i in rule]
    return sum(w * u[t] for w, t in terms), sum(abs(w * u[t]) for w, t in terms)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,lengths", [((5, 6, 7), (0, 1, 7, 8, 9)), ((9, 8, 11), (7, 16, 17, 64, 65, 125)),
                                           ((31, 17, 33), (1, 7, 7, 7, 33)), ((42, 40, 41), (7,))])
def test_grid_apply_rows(shape, lengths):
    import torch

    from jax_dips import _native as N
    from jax_dips.records import DeviceGrid, DeviceRecords, pack_dense

    rng = np.random.default_rng(3)
    n = int(np.prod(shape))
    ijk = np.stack(np.unravel_index(np.arange(n), shape), 1)
    W = np.zeros((n, 250))
    off = np.array([(c % 5 - 2, c // 5 % 5 - 2, c // 25 - 2) for c in range(125)])
    for r in range(n):
        pos = ijk[r] + off
        ok = np.nonzero(((pos >= -1) & (pos <= np.array(shape))).all(1))[0]  # the grid and its one ghost layer
        k = min(lengths[r % len(lengths)], len(ok))
        pick = rng.choice(ok, k, replace=False)
        W[r, 2 * pick + rng.integers(0, 2, k)] = rng.normal(size=k)
    c = rng.normal(size=n)
    axes = [np.linspace(-1, 1, m, dtype=np.float32) for m in shape]
    rec = DeviceRecords(pack_dense(W, c, n), np.full(3, 0.1, np.float32))
    grid = DeviceGrid(*axes)
    u = rng.normal(size=n).astype(np.float32)
    y = torch.zeros(n, dtype=torch.float32, device="cuda")
    ut = torch.as_tensor(u, device="cuda")
    for with_c in (0, 1):
        N.check(N.lib().dips_grid_apply(ctypes.byref(grid.c), ctypes.byref(rec.c), N.ptr(ut), N.ptr(y), with_c,
                                        N.current_stream()), "dips_grid_apply")
        got = y.cpu().numpy().astype(np.float64)
        ug = u.astype(np.float64).reshape(shape)
        for r in range(n):
            s, mag, L = (np.float64(np.float32(c[r])) if with_c else 0.0), abs(c[r]) * with_c, 0
            for q in np.nonzero(W[r])[0]:
                v, m = ghost(ug, ijk[r] + off[q // 2], shape)
                w = np.float64(np.float32(W[r, q]))
                s, mag, L = s + w * v, mag + abs(w) * m, L + 1
            assert abs(got[r] - s) <= 4 * (L + 1) * 2.0 ** -24 * mag + 1e-30, (r, got[r], s)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [6, 31, 33, 52])
def test_solve_sizes(n):
    """A quadratic solution, exact on the grid, from one workgroup of elements to a workspace shared with dead vectors."""
    from jax_dips.domain import mesh
    from jax_dips.judge import GridJudge

    mu = 2.5
    c = lambda v: (lambda r: r[0] * 0 + v)
    quad = lambda r: r[0] ** 2 + 2 * r[1] ** 2 - r[2] ** 2 + r[0] * r[1] + 0.3 * r[2]
    cbs = dict(phi=c(-1.0), mu_m=c(mu), mu_p=c(7.0), k_m=c(0.0), k_p=c(0.0), f_m=c(-mu * 4.0), f_p=c(0.0),
               alpha=c(0.0), beta=c(0.0), g=quad)
    gs = mesh.construct(3)[0](*problems.grid_axes(n))
    jd = GridJudge(gs, gs, cbs)
    u, it, rr = jd.solve(rtol=1e-6)
    assert 0 < it < 5000 and rr <= 1e-5
    res = jd.residual_vector(u)
    ref = jd.residual_vector(np.zeros_like(u))  # c
    assert np.linalg.norm(res) <= 1e-5 * np.linalg.norm(ref)
    # stopping early: exactly the iterations asked for, across the chunks the host waits for; none at all
    for k in (1, 7, 8, 9):
        if k < it:
            assert jd.solve(max_iter=k, rtol=0.0)[1] == k
    assert jd.solve(x0=u, rtol=1e-3)[1] == 0 and jd.solve(max_iter=0)[1] == 0
    # the same solve again: the same bits
    assert np.array_equal(jd.solve(rtol=1e-6)[0], u)
