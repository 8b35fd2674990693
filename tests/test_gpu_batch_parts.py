"""Batched training steps whose blocks are summed in parts (many tiles per block).

Whether a block's parts are one work item or several depends on the persistent grid's size and on the other problems;
the result must not: bit for bit.  Against the single-problem engine the sums of the first step differ in float32
order only (1e-5 relative on the loss, as for the tile kernel against its oracle).
"""
import numpy as np
import pytest

from helpers import oracle_level
from jax_dips import problems
from oracle import mlp as M

CFG = {"optimizer_name": "custom", "learning_rate": 1e-2,
       "sched": {"scheduler_name": "exponential", "decay_rate": 0.9}}


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(1, 1, 2, 10), (2, 16, 2, 16)])
@pytest.mark.parametrize("cap", [2, 3])
def test_parts_do_not_depend_on_the_grid_or_the_other_problems(dims, cap):
    from jax_dips.records import BatchEngine, DeviceGrid, DeviceRecords, Engine, pack_dense
    import torch

    levels = []
    for prob, n, batch in ((problems.sphere(mu_m=2.0, mu_p=7.0), 16, 4096), (problems.sphere(), 12, 640),
                           (problems.sphere(mu_p=3.0), 14, 2744)):
        axes, P, h, bounds, cb, rec = oracle_level(prob, n, 1)
        levels.append((DeviceGrid(*axes), DeviceRecords(pack_dense(rec.W, rec.c, batch), rec.h), batch))
    params = [M.init_params(dims, seed=70 + i) for i in range(3)]

    def run(which, grid_blocks, epochs=3):
        be = BatchEngine(dims, [params[i] for i in which], CFG, [64] * len(which))
        be.train_level([levels[i][0] for i in which], [levels[i][1] for i in which], epochs, cfg=(cap, grid_blocks))
        torch.cuda.synchronize()
        return [(e.params.cpu().numpy(), e.m.cpu().numpy(), e.v.cpu().numpy(), e.loss_hist.cpu().numpy(),
                 int(e.count.item())) for e in be.engines]

    ref = run((0, 1, 2), 0)
    for which, blocks in (((0, 1, 2), 1), ((0, 1, 2), 2), ((0, 1, 2), 5), ((0,), 1), ((0,), 64), ((2, 0), 3)):
        for i, got in zip(which, run(which, blocks)):
            for x, y in zip(ref[i], got):
                assert np.array_equal(x, y), (which, blocks, i)
    for i in range(3):
        eng = Engine(dims, params[i], CFG, max_rows=levels[i][2], max_steps=64)
        eng.train_level(levels[i][0], levels[i][1], 1)
        torch.cuda.synchronize()
        one = float(eng.loss_hist[0])
        assert abs(ref[i][3][0] - one) <= 1e-5 * abs(one)
        assert ref[i][4] == 3 * len(levels[i][1].batch_begin)
