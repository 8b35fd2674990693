"""The grid operator on the last entries that 32-bit row pointers can index (2^31 - 1 of them): rows of 7 beside
one of 33, whose rounds of 8 go on past the others' ends.  Tolerance as in test_gpu_judge_rows.py."""
import ctypes

import numpy as np
import pytest


@pytest.mark.gpu
def test_rows_at_the_end_of_the_index_range():
    import torch

    from jax_dips import _native as N
    from jax_dips.records import DeviceGrid, DeviceRecords

    rng = np.random.default_rng(0)
    nnz, n = 2 ** 31 - 1, 6
    rows = n ** 3
    axes = [np.linspace(-1, 1, n, dtype=np.float32)] * 3
    ijk = np.stack(np.unravel_index(np.arange(rows), (n, n, n)), 1)
    lengths = np.full(rows, 7)
    lengths[-40] = 33
    ptr = nnz - lengths.sum() + np.concatenate([[0], np.cumsum(lengths)])
    off = np.array([(c % 5 - 2, c // 5 % 5 - 2, c // 25 - 2) for c in range(125)])
    code = np.concatenate([rng.choice(np.nonzero(((ijk[r] + off >= 0) & (ijk[r] + off < n)).all(1))[0],
                                      min(lengths[r], 27)) for r in range(rows)])
    extra = np.full(lengths.sum() - code.size, 62)  # the row of 33: its own node for the rest
    at = int(lengths[:rows - 40].sum()) + 27
    code = np.insert(code, at, extra)
    w = rng.normal(size=code.size).astype(np.float32)
    u = rng.normal(size=rows).astype(np.float32)
    codes = torch.empty(nnz, dtype=torch.int32, device="cuda")
    weights = torch.empty(nnz, dtype=torch.float32, device="cuda")
    codes[nnz - code.size:] = torch.as_tensor(code.astype(np.int32), device="cuda")
    weights[nnz - code.size:] = torch.as_tensor(w, device="cuda")

    def T(a, dt):
        return torch.as_tensor(np.asarray(a), device="cuda").to(dt)

    c = rng.normal(size=rows).astype(np.float32)
    rec = DeviceRecords.from_device(T(np.arange(rows), torch.int32), T(ptr, torch.int32), T(c, torch.float32), codes,
                                    weights, nnz, np.full(3, 0.1, np.float32), rows, [0], [rows], [0])
    grid = DeviceGrid(*axes)
    y = torch.zeros(rows, dtype=torch.float32, device="cuda")
    N.check(N.lib().dips_grid_apply(ctypes.byref(grid.c), ctypes.byref(rec.c), N.ptr(T(u, torch.float32)), N.ptr(y), 1,
                                    N.current_stream()), "dips_grid_apply")
    got = y.cpu().numpy().astype(np.float64)
    begin = np.concatenate([[0], np.cumsum(lengths)])
    for r in range(rows):
        p = ijk[r] + off[code[begin[r]:begin[r + 1]]]
        t = w[begin[r]:begin[r + 1]].astype(np.float64) * u[(p[:, 0] * n + p[:, 1]) * n + p[:, 2]]
        assert abs(got[r] - (c[r] + t.sum())) <= (lengths[r] + 1) * 2.0 ** -24 * (abs(c[r]) + np.abs(t).sum()), r
