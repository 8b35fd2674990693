"""The chained two-layer 16-wide tile step with many tiles per wavefront: a wavefront takes its tiles in windows of 64,
first those with + entries, then those with - entries, and the rows of more than 64 entries at the end, which it finds by a
mask in the first window and by their length after it.

One block of 8 wavefronts sums a batch of about 2900 tiles in four parts, 90 tiles a wavefront and part, with long rows
and empty ones all over the batch.  Loss and gradient (as the first moment of one clipped step) against float64 autograd: 1e-5 and
1e-4 (2-norm), as in test_gpu_tile_chain.py.
"""
import numpy as np
import pytest


def batch(seed):
    """Rows of 9 random entries: + only, - only, or both; one in 400 of 65 to 130 entries, one in 300 empty; not sorted."""
    rng = np.random.default_rng(seed)
    n = 27
    rows = n ** 3
    lengths = np.full(rows, 9)
    lengths[rng.random(rows) < 1 / 400] = -1
    lengths[lengths < 0] = rng.integers(65, 131, int((lengths < 0).sum()))
    lengths[rng.random(rows) < 1 / 300] = 0
    share = np.repeat([1.0, 0.0, 0.5], -(-rows // 3))[:rows]
    ptr = np.concatenate([[0], np.cumsum(lengths)])
    row = np.repeat(np.arange(rows), lengths)
    code = rng.integers(0, 125, row.size) | ((rng.random(row.size) < share[row]).astype(np.int64) << 7)
    packed = dict(row_point=rng.permutation(rows).astype(np.int32), row_ptr=ptr.astype(np.int32),
                  row_c=rng.normal(size=rows).astype(np.float32), ent_code=code.astype(np.uint32),
                  ent_w=(rng.normal(size=row.size) / np.sqrt(lengths[row])).astype(np.float32), batch_size=rows,
                  batch_begin=[0], batch_rows=[rows], batch_nbulk=[0])
    return n, packed, lengths


def reference(grid, rec, theta, act):
    import torch

    th = theta.double().requires_grad_(True)
    ptr = rec.row_ptr.long()
    row = torch.repeat_interleave(torch.arange(rec.nrows, device="cuda"), ptr[1:] - ptr[:-1])
    code = rec.ent_code[:rec.nnz].long()
    k = code & 127
    o = torch.stack([k % 5 - 2, k // 5 % 5 - 2, k // 25 - 2], 1).float()
    x = (grid.points()[rec.row_point.long()[row]] + o * torch.as_tensor(rec.h, device="cuda")).double()
    u, off = [], 0
    for _ in range(2):
        a = x
        for i, (m, n) in enumerate(((3, 16), (16, 16), (16, 1))):
            a = a @ th[off:off + m * n].view(m, n) + th[off + m * n:off + m * n + n]
            off += m * n + n
            if i < 2:
                a = torch.nn.functional.celu(a) if act else torch.tanh(a)
        u.append(a[:, 0])
    v = torch.where((code & 128) != 0, u[0], u[1]) * rec.ent_w[:rec.nnz].double()
    r = rec.row_c.double().index_add(0, row, v)
    loss = 0.5 * (r * r).sum() / rec.nrows
    (g,) = torch.autograd.grad(loss, th)
    return loss.item(), g


@pytest.mark.gpu
@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("cap", [1, 256])
def test_many_tiles_per_wavefront(act, cap):
    import torch

    from jax_dips.records import BatchEngine, DeviceGrid, DeviceRecords

    n, packed, lengths = batch(act)
    grid = DeviceGrid(*[np.linspace(-1, 1, n, dtype=np.float32)] * 3)
    rec = DeviceRecords(packed, np.full(3, 0.037, np.float32))
    tiles = int(np.diff(rec.tiles(grid)["batch_tile_begin"])[0]) - 1
    long = np.nonzero(lengths > 64)[0]
    assert tiles > 4 * 8 * 80 and len(long) > 20 and (lengths == 0).sum() > 20
    g = torch.Generator().manual_seed(act)
    parts = []
    for _ in range(2):
        for a, b in ((3, 16), (16, 16), (16, 1)):
            parts += [torch.randn(a * b, generator=g) / a ** 0.5, 0.1 * torch.randn(b, generator=g)]
    theta = torch.cat(parts)
    be = BatchEngine((2, 16, 2, 16), [theta.numpy()], {"optimizer_name": "custom", "learning_rate": 1e-3,
                     "sched": {"scheduler_name": "exponential", "decay_rate": 0.9}}, [4], act=act)
    be.train_level([grid], [rec], 1, cfg=(cap, 0))
    torch.cuda.synchronize()
    loss, want = reference(grid, rec, theta.cuda(), act)
    e = be.engines[0]
    want = 0.1 * want / max(1.0, float(want.norm()))
    assert abs(float(e.loss_hist[0]) - loss) <= 1e-5 * loss
    assert float((e.m.double() - want).norm()) <= 1e-4 * float(want.norm())
