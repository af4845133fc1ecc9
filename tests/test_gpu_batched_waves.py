"""Batched launches whose wave counts are no multiple of the workgroup size: every
work item runs, whatever number of whole workgroups the waves make."""
import numpy as np
import pytest

from conftest import haar_state

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _batch(rng, rows, per_row):
    import mentpy_amd as mp
    from mentpy_amd.batched import BatchedForward
    jobs = []
    for r in rows:
        for i in range(per_row):
            g = mp.templates.grid_cluster(r, 4 + i % 3)
            th = rng.uniform(0, 2 * np.pi, (1000, len(g.trainable_nodes))).astype(np.float32)
            jobs.append((mp.PatternSimulator(g, backend="hip-sv"), th, haar_state(r, rng)[None]))
    return BatchedForward(jobs, sims_per_item=64)


# (waves, wg_waves): whole workgroups make 4, 30, 3 and 60 waves of them
@pytest.mark.parametrize("waves,wg_waves", [(6, 4), (32, 3), (5, 3), (63, 4)])
@pytest.mark.parametrize("rows", [(3,), (2, 3, 4)])
def test_every_item_runs(rows, waves, wg_waves, rng):
    """Outputs filled with NaN equal a launch of one-wave workgroups bit for bit: all
    groups together, and each group with that many waves of its own."""
    torch = _torch()
    from mentpy_amd.batched import MAX_GROUPS
    bf = _batch(rng, rows, 4)
    want = [o.clone() for o in bf.launch(waves=256, wg_waves=1)]
    for kw in ({"waves": waves}, {"group_waves": [waves] * MAX_GROUPS}):
        for o in bf.outputs:
            o.fill_(complex(float("nan"), 0.0))
        got = bf.launch(wg_waves=wg_waves, **kw)
        torch.cuda.synchronize()
        for x, y in zip(got, want):
            assert torch.equal(x, y), kw
