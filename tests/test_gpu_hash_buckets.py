"""The rows of a table over the buckets of its gradient: tables of one bucket and of several, without dense levels,
without hashed ones, with level sizes that are no multiple of a bucket's row groups.  Loss and gradient of a batch
against the float64 oracle at the tolerances of the other hashgrid tests; every row's gradient lands in its row, so
rows that no entry touches are exactly zero.
"""
import numpy as np
import pytest

from helpers import oracle_level
from jax_dips import problems
from oracle import hashgrid as HG
from test_gpu_hashgrid import _model, _rel

TABLES = {
    "one bucket": {"pos_levels": 3, "T": 1000, "N_min": 4, "N_max": 24},
    "odd sizes": {"pos_levels": 6, "T": 12347, "N_min": 5, "N_max": 90},
    "all dense": {"pos_levels": 3, "T": 2 ** 19, "N_min": 9, "N_max": 61},
    "first level hashed": {"pos_levels": 4, "T": 501, "N_min": 8, "N_max": 40},
    "many buckets": {"pos_levels": 12, "T": 2 ** 17, "N_min": 16, "N_max": 512},
    # upper-face points index past the last dense level's rows, into the next level's; 256 slots a workgroup, none full
    "past a dense level": {"pos_levels": 12, "T": 2 ** 17, "N_min": 16, "N_max": 540},
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(TABLES))
def test_table_gradient_rows(name):
    from jax_dips.records import DeviceGrid, DeviceRecords, HashEngine, pack_dense

    B = 2048
    axes, P, h, bounds, cb, rec = oracle_level(problems.sphere(mu_m=1.0, mu_p=10.0), 16, 1)
    model, theta, grid, n_mlp = _model(TABLES[name], 4, 1e4)
    eng = HashEngine(model.hashgrid, theta, {}, max_steps=2)
    dgrid, drec = DeviceGrid(*axes), DeviceRecords(pack_dense(rec.W, rec.c, B), rec.h)
    loss, grad = eng.loss_grad(dgrid, drec, 1, 1.0 / B)
    ol, og, _ = HG.loss_and_grad(theta.astype(np.float64), grid, [16], rec, np.arange(B, 2 * B))
    assert abs(loss - ol) <= 1e-5 * abs(ol)
    assert _rel(grad[:n_mlp], og[:n_mlp]) <= 1e-4 and _rel(grad[n_mlp:], og[n_mlp:]) <= 1e-4
    assert np.array_equal(grad[n_mlp:] == 0, og[n_mlp:] == 0)
