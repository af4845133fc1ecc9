"""Both sides of the lines between kernels of the same launch: the results are the same
bit for bit where the kernels promise it, else within a bound of the oracle."""
import numpy as np
import pytest

from conftest import haar_state

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _sim(rows, cols, window=None):
    import mentpy_amd as mp
    g = mp.templates.grid_cluster(rows, cols)
    return g, mp.PatternSimulator(g, backend="hip-sv", **({"window_size": window} if window else {}))


@pytest.mark.parametrize("rows,cols,window", [(2, 12, None), (3, 8, None), (2, 9, 4), (1, 9, 3)])
@pytest.mark.parametrize("B", [512, 513])
def test_two_and_three_slots_either_side_of_512(rows, cols, window, B, rng):
    """2 and 3 slots share coefficients between lanes up to 512 simulations: row by row
    equal to a small launch, and the oracle's amplitudes."""
    torch = _torch()
    from oracle.vectorized import sv_batch
    g, sim = _sim(rows, cols, window)
    assert sim.simulator.plan.info["n_slots"] in (2, 3)
    gen = torch.Generator().manual_seed(rows * cols)
    th = (torch.rand((B, len(g.trainable_nodes)), generator=gen) * 12 - 6).cuda()
    psi = haar_state(rows, rng)
    full = sim.run_batch(th, psi)
    for part in (slice(0, 9), slice(B - 9, B)):
        assert torch.equal(full[part], sim.run_batch(th[part].contiguous(), psi))
    ref = sv_batch(g, th[-8:].double().cpu().numpy(), psi[None])
    assert np.abs(full[-8:].cpu().numpy() - ref).max() < 2e-5
