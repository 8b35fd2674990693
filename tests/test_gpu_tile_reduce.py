"""The optimizer workgroup of a tile training step: its float64 sums over the workgroups' partial rows.

One step from zero moments leaves m = 0.1 g (Adam, b1 = 0.9), clipped as a whole, so m / |m| is the direction of the
gradient that the step reduced; dips_tile_loss_grad reduces the same rows through a kernel of its own.  Both are
float64 sums of equal float32 rows rounded once (2^-24 of an entry) and scaled: 1e-6 of the norm, and 1e-6 of the
loss, cover the roundings.  The batches give 1 row, fewer rows than row groups, a remainder of the rows in flight
and the most rows; the shapes one, two and three wavefronts per row.
"""
import numpy as np
import pytest

from helpers import oracle_level
from jax_dips import problems
from oracle import mlp as M

CFG = {"optimizer_name": "custom", "learning_rate": 1e-2,
       "sched": {"scheduler_name": "exponential", "decay_rate": 0.9}}


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(1, 1, 1, 1), (2, 10, 2, 10), (2, 16, 2, 16)])
@pytest.mark.parametrize("n,batch", [(12, 64), (12, 300), (16, 4096), (28, 28 ** 3)])
def test_step_reduces_the_rows_of_loss_grad(dims, n, batch):
    from ctypes import byref

    from jax_dips import _native as N
    from jax_dips.records import DeviceGrid, DeviceRecords, Engine, pack_dense
    import torch

    axes, P, h, bounds, cb, rec = oracle_level(problems.sphere(mu_m=2.0, mu_p=7.0), n, 1)
    grid, drec = DeviceGrid(*axes), DeviceRecords(pack_dense(rec.W, rec.c, batch), rec.h)
    theta = M.init_params(dims, seed=8)
    eng = Engine(dims, theta, CFG, max_rows=batch, max_steps=4096)
    loss, grad = eng.tile_loss_grad(grid, drec, 0, 1.0 / batch)
    for single in (False, True):
        e = Engine(dims, theta, CFG, max_rows=batch, max_steps=4096)
        e.tile_single_launch = single
        tl = drec.tiles(grid)
        tb = tl["batch_tile_begin"]
        N.check(N.lib().dips_tile_train_step(
            byref(grid.c), byref(drec.c), byref(tl["c"]), int(tb[0]), int(tb[1] - tb[0] - 1), byref(e.net),
            byref(e.opt), 1.0 / batch, N.ptr(e.params), N.ptr(e.m), N.ptr(e.v), N.ptr(e.count), N.ptr(e.loss_hist),
            int(e.loss_hist.numel()), N.ptr(e.partial), e.partial_cap, N.ptr(e.sync) if single else None,
            N.current_stream()), "dips_tile_train_step")
        torch.cuda.synchronize()
        m = e.m.cpu().numpy().astype(np.float64)
        assert abs(float(e.loss_hist[0]) - loss) <= 1e-6 * abs(loss)
        d = m / np.linalg.norm(m) - grad / np.linalg.norm(grad)
        assert np.linalg.norm(d) <= 1e-6, (single, np.linalg.norm(d))
        assert int(e.count.item()) == 1
