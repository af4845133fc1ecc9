"""Density matrices at the batches where the kernels change: the matrix kernels of plans off
the column structure (one entry per lane, LDS, one simulation per lane) and the
Pauli-vector kernels of column plans, against the oracle and against the general
kernel that evaluates every step's probability."""
import numpy as np
import pytest

from conftest import haar_state

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


# (rows, cols, window, slots, column plan, angle vectors, inputs)
CASES = [(1, 7, None, 1, True, 32768, 1), (1, 7, None, 1, True, 32769, 1),
         (1, 8, 3, 2, False, 8192, 2), (1, 8, 3, 2, False, 16385, 1), (1, 8, 3, 2, False, 40000, 1),
         (2, 5, 4, 3, False, 1024, 1), (2, 5, 4, 3, False, 1025, 1), (2, 5, 4, 3, False, 32767, 1),
         (2, 5, 4, 3, False, 16384, 2), (2, 5, 4, 3, False, 40001, 1),
         (3, 4, None, 3, True, 12288, 4), (2, 5, None, 2, True, 16384, 3), (4, 4, None, 4, True, 2048, 1),
         (4, 4, None, 4, True, 2049, 1)]


@pytest.mark.parametrize("rows,cols,window,slots,column,B,S", CASES)
def test_dm_kernels_by_batch(rows, cols, window, slots, column, B, S, rng):
    """Amplitudes of a sample within 2e-5 of the oracle (single precision over a few dozen
    steps), every simulation within 2e-5 of the step-probability kernel, which shares no
    code with them, and nothing stored past the last matrix."""
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.noise import NoiseModel
    from mentpy_amd.simulators.hip_simulator import dm_forward
    from oracle.vectorized import dm_batch
    g = mp.templates.linear_cluster(cols) if rows == 1 else mp.templates.grid_cluster(rows, cols)
    sim = mp.PatternSimulator(g, backend="hip-dm", **({"window_size": window} if window else {}))
    plan = sim.simulator.plan
    assert plan.info["n_slots"] == slots and bool(plan.info["periodic"]) is column
    th = rng.uniform(-7, 7, (B, len(g.trainable_nodes))).astype(np.float32)
    psi = np.stack([haar_state(rows, rng) for _ in range(S)])
    a = torch.as_tensor(th, device="cuda")
    s = torch.as_tensor(psi, dtype=torch.complex64, device="cuda")
    d = 1 << rows
    noise = NoiseModel(depolarizing=0.03, readout_flip=0.01)
    guard = torch.full((B + 1, S, d, d), 7.0, dtype=torch.complex64, device="cuda")
    out = dm_forward(plan, a, s, noise=noise, out=guard[:B])
    general = dm_forward(plan, a, s, noise=noise, step_probs=True)
    torch.cuda.synchronize()
    assert (guard[B] == 7.0).all()
    assert (out - general).abs().max().item() < 2e-5
    at = [0, B // 2, B - 1]
    ref = dm_batch(g, th[at].astype(np.float64), psi, p_depol=0.03, p_readout=0.01)
    assert np.abs(out[at].cpu().numpy() - ref).max() < 2e-5
