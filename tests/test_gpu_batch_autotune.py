"""What the batch autotuner measures and what it takes from its file: every timed step trains every problem, also where a
problem has one batch; entries of another build of the library, or of other tiles per batch, are not used."""
import json

import numpy as np
import pytest

from helpers import oracle_level
from jax_dips import problems
from oracle import mlp as M

CFG = {"optimizer_name": "custom", "learning_rate": 1e-2,
       "sched": {"scheduler_name": "exponential", "decay_rate": 0.9}}
DIMS = (2, 16, 2, 16)


def level(n, zoom, batch):
    from jax_dips.records import DeviceGrid, DeviceRecords, pack_dense

    axes, P, h, bounds, cb, rec = oracle_level(problems.sphere(mu_m=2.0, mu_p=7.0), n, zoom)
    return DeviceGrid(*axes), DeviceRecords(pack_dense(rec.W, rec.c, batch), rec.h)


@pytest.mark.gpu
def test_every_timed_step_trains_every_problem(tmp_path, monkeypatch):
    from jax_dips import records
    from jax_dips.records import BatchEngine
    import torch

    levels = [level(12, 1, 1728), level(10, 1, 500)]  # one batch, two batches
    grids, recs = [g for g, _ in levels], [r for _, r in levels]
    be = BatchEngine(DIMS, [M.init_params(DIMS, seed=i) for i in range(2)], CFG, [64] * 2)
    trained = []
    restore = be._restore
    monkeypatch.setattr(be, "_restore", lambda snap: (trained.append([int(e.count.item()) for e in be.engines]),
                                                      restore(snap)))
    records._BATCH_TUNED.clear()
    be.autotune(grids, recs, caps=(256, 16), steps=6, cache_path=str(tmp_path / "tune.json"))
    assert trained == [[7, 7]] * 4  # a warm-up step and six timed ones, of each candidate
    torch.cuda.synchronize()
    assert [int(e.count.item()) for e in be.engines] == [0, 0]


@pytest.mark.gpu
def test_file_entries_of_other_builds_and_levels_are_not_used(tmp_path, monkeypatch):
    from jax_dips import _native as N
    from jax_dips import records
    from jax_dips.records import BatchEngine

    path = str(tmp_path / "tune.json")

    def tune(zoom, revision=None):
        g, r = level(12, zoom, 600)
        be = BatchEngine(DIMS, [M.init_params(DIMS, seed=1)], CFG, [64])
        records._BATCH_TUNED.clear()
        with monkeypatch.context() as m:
            if revision:
                m.setattr(N, "library_revision", lambda: revision)
            cfg = be.autotune([g], [r], caps=(256, 16), steps=2, cache_path=path)
        return cfg, hasattr(be, "tuning")

    assert tune(1, "another build")[1]
    disk = {k: {"cfg": [3, 5]} for k in json.load(open(path))}
    json.dump(disk, open(path, "w"))
    assert tune(1, "another build") == ((3, 5), False)
    cfg, measured = tune(1)
    assert measured and cfg != (3, 5)
    assert tune(1) == (cfg, False)  # its own entry
    assert tune(3)[1]  # the same points and batch size, other tiles
    assert len(json.load(open(path))) == 3
