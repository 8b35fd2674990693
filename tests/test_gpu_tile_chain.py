"""Loss and gradient of the two-layer 13..16-wide tile networks (chained matrix products over 16-slot sub-tiles)
against the float64 oracle: tiles of one and of both phases, rows of more than 64 entries and empty ones, part-filled
last tiles.  float32 networks and sums: 1e-5 relative on the loss, 1e-4 (2-norm) on the gradient, as for the other shapes.
"""
import numpy as np
import pytest

from helpers import oracle_level
from jax_dips import problems
from oracle import mlp as M
from oracle import trainer as T


@pytest.mark.gpu
@pytest.mark.parametrize("level,long", [(0, False), (1, False), (2, True)])
@pytest.mark.parametrize("n,batch", [(12, 61), (12, 1728), (16, 4096)])
def test_chain_loss_grad(level, long, n, batch):
    from jax_dips.records import DeviceGrid, DeviceRecords, Engine, pack_dense
    from test_gpu_tiles import _synthetic_long_rows

    dims = (2, 16, 2, 16)
    axes, P, h, bounds, cb, rec = oracle_level(problems.sphere(mu_m=2.0, mu_p=7.0, k_m=0.5, k_p=1.5), n, level)
    if long:
        rec, _ = _synthetic_long_rows(rec, 5)
    grid, drec = DeviceGrid(*axes), DeviceRecords(pack_dense(rec.W, rec.c, batch), rec.h)
    theta = M.init_params(dims, seed=5)
    eng = Engine(dims, theta, {}, max_rows=batch, max_steps=4)
    assert int((drec.row_ptr[1:] - drec.row_ptr[:-1] > 64).sum()) > 0 or not long
    for b in sorted({0, len(drec.batch_begin) // 2, len(drec.batch_begin) - 1}):
        b0, nrow = int(drec.batch_begin[b]), int(drec.batch_rows[b])
        rows = drec.row_point[b0:b0 + nrow]
        rows = np.asarray(rows.cpu() if hasattr(rows, "cpu") else rows)
        loss, grad = eng.tile_loss_grad(grid, drec, b, 1.0 / nrow)
        ol, og, _ = T.loss_and_grad(theta.astype(np.float64), dims, rec, rows)
        assert abs(loss - ol) <= 1e-5 * abs(ol), (b, loss, ol)
        assert np.linalg.norm(grad - og) <= 1e-4 * np.linalg.norm(og), b
