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


def _tile_jobs(rng, n, specs):
    import mentpy_amd as mp
    jobs = []
    for i in range(n):
        rows, cols, window, sets, inputs = specs[i % len(specs)]
        g = mp.templates.grid_cluster(rows, cols)
        sim = mp.PatternSimulator(g, backend="hip-sv", **({"window_size": window} if window else {}))
        th = rng.uniform(-7, 7, (sets, len(g.trainable_nodes))).astype(np.float32)
        jobs.append((sim, th, np.stack([haar_state(rows, rng) for _ in range(inputs)])))
    return jobs


# (rows, cols, window, angle vectors, inputs); windows of rows + 2 and more give plans off
# the column structure with rows + 1 slots and more, whose last blocks are partial
@pytest.mark.parametrize("n,specs", [
    (5, [(15, 4, None, 1, 1), (15, 3, None, 2, 1), (15, 5, None, 1, 2)]),    # uneven lengths
    (5, [(15, 3, None, 1, 1), (4, 6, 16, 3, 1), (2, 9, 16, 1, 2)]),          # off the column structure
    (44, [(4, 6, 16, 4, 1), (3, 7, 16, 2, 1), (5, 5, 16, 3, 1)]),            # 132 simulations: two chunks
    (6, [(16, 3, None, 1, 1), (5, 6, 17, 1, 2), (15, 3, None, 1, 1), (17, 3, None, 1, 1)]),
])
def test_wide_jobs_run_together(n, specs, rng):
    """Groups of 15 slots and more take the simulations of all their jobs in the same
    passes: every job equals its own launch bit for bit, also from the tables, in
    the raw phase and replayed from a graph."""
    torch = _torch()
    from mentpy_amd.batched import BatchedForward
    jobs = _tile_jobs(rng, n, specs)
    bf = BatchedForward(jobs, sims_per_item=64)
    assert max(bf.groups()) >= 15
    for kw in ({}, {"table_steps": True}, {"ref_phase": False, "renormalize": False}):
        for o in bf.outputs:
            o.fill_(complex(float("nan"), 0.0))
        got = bf.launch(waves=64, wg_waves=1, **kw)
        single = {} if "ref_phase" not in kw else {"phase": "raw", "renormalize": False}
        torch.cuda.synchronize()
        for (sim, th, st), o in zip(jobs, got):
            assert torch.equal(sim.run_batch(th, st, **single), o), kw
    want = [o.clone() for o in bf.launch(waves=64, wg_waves=1)]
    graph = bf.capture_graph(waves=64, wg_waves=1)
    for _ in range(3):
        for o in bf.outputs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, w) for o, w in zip(bf.outputs, want))


def test_many_wide_jobs_fill_the_chip(rng):
    """64 jobs of one simulation each take little longer than one of them, which leaves most
    of the chip idle (one job after the other: 64 times as long and more)."""
    torch = _torch()
    from mentpy_amd.batched import BatchedForward

    def best(n):
        bf = BatchedForward(_tile_jobs(rng, n, [(15, 4, None, 1, 1)]))
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        times = []
        for _ in range(10):
            start.record()
            bf.launch()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    one, many = best(1), best(64)
    print(f"one job {one * 1e3:.0f} us, 64 jobs {many * 1e3:.0f} us", flush=True)
    assert many < 16 * one
