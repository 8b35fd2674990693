"""The table gradient where its record slots decide it: slots of several chunks of 256 records, full, part-filled and
empty ones, small tables spread over more buckets than their rows need (and, at the smaller batches, not).

A batch's gradient is the sum of its rows' (each row's residual depends on the parameters only), so a large batch is
compared with small ones, whose few records per slot test_gpu_hash_buckets.py compares with the float64 oracle.  Every
float32 value is within 2^-24 of its sum, of the MLPs' partial sums within 1e-6: 1e-5 (2-norm).
"""
import numpy as np
import pytest

from test_gpu_mfma_split import records

TABLES = {"one dense level": (2, 2, 4096, 4, 16, 1.0, 0), "2^14": (16, 2, 1 << 14, 16, 2048, 1.0, 0),
          "odd": (8, 2, 12347, 5, 900, 1.0, 0), "2^19": (16, 2, 1 << 19, 16, 2048, 1.0, 0)}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(TABLES))
@pytest.mark.parametrize("rows,per_row", [(300, 3), (30000, 9)])
def test_gradient_of_many_records_per_slot(name, rows, per_row):
    import torch

    from jax_dips import _native as N
    from jax_dips.records import DeviceGrid, DeviceRecords, HashEngine

    grid, big = records(rows, per_row, 0.4, rows)
    grid = DeviceGrid(*[np.linspace(-0.9, 0.9, n, dtype=np.float32) for n in grid.shape])  # every entry inside the box
    host = {k: np.asarray(getattr(big, k).cpu()) for k in ("row_point", "row_ptr", "row_c", "ent_code", "ent_w")}
    P = int(N.lib().dips_hash_param_count(N.HashGrid(*TABLES[name])))
    g = torch.Generator().manual_seed(rows)
    eng = HashEngine(TABLES[name], (0.2 * torch.randn(P, generator=g)).numpy(), {}, max_steps=2)
    n_mlp = P - 2 * int(N.lib().dips_hash_table_rows(N.HashGrid(*TABLES[name])))
    loss, grad = eng.loss_grad(grid, big, 0, 1.0)
    total, want = 0.0, np.zeros(P)
    B = max(100, rows // 12)
    begin = np.arange(0, rows, B)
    small = DeviceRecords(dict(host, batch_size=B, batch_begin=begin, batch_rows=np.minimum(B, rows - begin),
                               batch_nbulk=np.zeros(len(begin), np.int64)), big.h)
    eng._work = None
    for b in range(len(begin)):
        l1, g1 = eng.loss_grad(grid, small, b, 1.0)
        total, want = total + l1, want + g1
    assert abs(loss - total) <= 1e-6 * abs(total)
    for part in (slice(0, n_mlp), slice(n_mlp, P)):
        assert np.linalg.norm(grad[part] - want[part]) <= 1e-5 * np.linalg.norm(want[part])
    assert np.array_equal(grad[n_mlp:] == 0, want[n_mlp:] == 0)
