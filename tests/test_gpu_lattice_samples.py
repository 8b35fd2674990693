"""The record build's list of distinct sample positions on the GPU (a bit per lattice point) against the sorted keys on
the host: the same positions in the same order, and the same values at every sample.  phi is a linear form in float64,
whose products and sums round alike on both.  Axes of 2 nodes, lattice rows of part of a word, of whole words
and of more words than a wavefront has lanes; coinciding and distinct coordinates; extra points.
"""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 2, 2), (5, 3, 11), (3, 7, 64), (2, 3, 300)])
@pytest.mark.parametrize("level", [0, 1, 3])
def test_lattice_samples_equal_sorted_keys(shape, level):
    import torch

    from jax_dips.level_records import STENCIL, stencil_corner_phi
    from jax_dips.records import DeviceGrid

    rng = np.random.default_rng(level)
    axes = [np.linspace(-1.0, 1.0, n, dtype=np.float32) for n in shape]
    h = np.array([(a[1] - a[0]) * np.float32(0.5) ** level for a in axes], np.float32)
    extra = rng.uniform(-1, 1, (5, 3))
    asked, got = [], []
    for device in ("cpu", "cuda"):
        grid = DeviceGrid(*axes, extra=extra, device=device)
        ht = torch.tensor(h, device=device)
        positions = []

        def phi(r):
            positions.append(r.cpu())
            return r[0] * 3.0 + r[1] * 5.0 - r[2] * 7.0

        P = grid.points()
        S = P[:, None, :] + torch.tensor(STENCIL, dtype=torch.float32, device=device)[None] * ht
        got.append([t.cpu() for t in stencil_corner_phi(grid, S, ht, ht * 0.5, phi)])
        asked.append(positions)
    assert len(asked[0]) == len(asked[1]) and all(torch.equal(a, b) for a, b in zip(*asked))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
