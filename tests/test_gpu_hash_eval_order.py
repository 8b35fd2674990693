"""dips_hash_eval has two loop orders of the MLP, chosen by the table's rows and the number of points: the same sums, so
the same bits for the same points in calls on either side of the line (rows times points: 2^43)."""
import ctypes

import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("levels", [16, 12])
def test_eval_bits_do_not_depend_on_the_call_size(levels):
    import torch

    from jax_dips import _native as N

    L = N.lib()
    hg = N.HashGrid(levels, 2, 1 << 19, 16, 2048, 1.0, 0)
    g = torch.Generator().manual_seed(levels)
    theta = (0.2 * torch.randn(int(L.dips_hash_param_count(ctypes.byref(hg))), generator=g)).cuda()
    m, part = 2000077, 1 << 19
    rows = L.dips_hash_table_rows(ctypes.byref(hg))
    assert rows * m >= 1 << 43 > rows * part
    pts = (2 * torch.rand(m, 3, generator=g) - 1).cuda()
    phase = (torch.rand(m, generator=g) < 0.5).to(torch.uint8).cuda()

    def run(a, b):
        u, gr = torch.empty(b - a, device="cuda"), torch.empty(b - a, 3, device="cuda")
        N.check(L.dips_hash_eval(ctypes.byref(hg), N.ptr(theta), N.ptr(pts[a:b].contiguous()),
                                 N.ptr(phase[a:b].contiguous()), b - a, N.ptr(u), N.ptr(gr), N.current_stream()),
                "dips_hash_eval")
        torch.cuda.synchronize()
        return u, gr

    u, gr = run(0, m)
    for a in range(0, m, part):
        b = min(m, a + part)
        u1, gr1 = run(a, b)
        assert torch.equal(u1, u[a:b]) and torch.equal(gr1, gr[a:b])
