"""More problems than the 64 lanes that write a step's item table, with different numbers of batches and steps: every one of
them follows its single-problem run bit for bit."""
import numpy as np
import pytest

from helpers import oracle_level
from jax_dips import problems
from oracle import mlp as M

CFG = {"optimizer_name": "custom", "learning_rate": 1e-2,
       "sched": {"scheduler_name": "exponential", "decay_rate": 0.9}}
DIMS = (1, 1, 2, 10)


@pytest.mark.gpu
@pytest.mark.parametrize("count", [64, 65, 130])
def test_more_problems_than_lanes(count):
    from jax_dips.records import BatchEngine, DeviceGrid, DeviceRecords, Engine, pack_dense
    import torch

    sets = []
    for n, batch in ((6, 216), (7, 100), (8, 512)):
        axes, P, h, bounds, cb, rec = oracle_level(problems.sphere(mu_m=2.0, mu_p=7.0), n, 1)
        sets.append((DeviceGrid(*axes), DeviceRecords(pack_dense(rec.W, rec.c, batch), rec.h), batch))
    pick = [sets[i % 3] for i in range(count)]
    params = [M.init_params(DIMS, seed=i) for i in range(count)]
    be = BatchEngine(DIMS, params, CFG, [16] * count)
    be.train_level([p[0] for p in pick], [p[1] for p in pick], 2)
    torch.cuda.synchronize()
    for i in (0, 1, 2, 62, 63, count - 2, count - 1):
        grid, rec, batch = pick[i]
        eng = Engine(DIMS, params[i], CFG, max_rows=batch, max_steps=16)
        eng.train_level(grid, rec, 2)
        torch.cuda.synchronize()
        got = be.engines[i]
        assert int(got.count.item()) == 2 * len(rec.batch_begin)
        for a, b in ((got.params, eng.params), (got.m, eng.m), (got.v, eng.v), (got.loss_hist, eng.loss_hist)):
            assert torch.equal(a, b), i
