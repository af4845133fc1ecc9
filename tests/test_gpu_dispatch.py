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


# (rows, cols, B, S): the raw-phase batches where the longest patterns of 4, 5 and 6 slots
# stop sharing coefficients between inputs, and where shorter ones still do
@pytest.mark.parametrize("rows,cols,B,S", [
    (4, 34, 7168, 4), (4, 34, 7169, 4), (4, 33, 8192, 4), (4, 33, 8193, 4),
    (5, 27, 3584, 8), (5, 27, 3585, 8), (5, 26, 4096, 8),
    (6, 13, 8192, 16), (6, 14, 3072, 16), (6, 14, 3073, 16), (6, 42, 2560, 16), (6, 42, 2561, 16)])
def test_shared_coefficients_by_steps(rows, cols, B, S):
    """Either side of the largest shared batches of short, longer and long patterns: equal
    to the launches of one input each."""
    torch = _torch()
    from mentpy_amd.simulators.hip_simulator import sv_forward
    g, sim = _sim(rows, cols)
    plan = sim.simulator.plan
    gen = torch.Generator().manual_seed(rows * cols)
    th = (torch.rand((B, len(g.trainable_nodes)), generator=gen) * 12 - 6).cuda()
    x = torch.randn((S, 1 << rows), generator=gen, dtype=torch.complex64).cuda()
    got = sv_forward(plan, th, x, ref_phase=False, renormalize=False)
    for i in (0, S - 1):
        one = sv_forward(plan, th[-64:], x[i:i + 1], ref_phase=False, renormalize=False)
        assert torch.equal(got[-64:, i], one[:, 0])
        one = sv_forward(plan, th[:64], x[i:i + 1], ref_phase=False, renormalize=False)
        assert torch.equal(got[:64, i], one[:, 0])


# (rows, cols, columns per set, sets): the last batch of the sweeps that spread a
# simulation over lanes and the first one above it
@pytest.mark.parametrize("rows,cols,C,B", [
    (4, 6, 3, 8192), (4, 6, 3, 8193), (4, 42, 1, 16384), (4, 42, 1, 16385), (4, 6, 16, 2048),
    (4, 6, 16, 2049), (5, 5, 3, 15018), (5, 5, 3, 15019), (5, 5, 16, 2560), (5, 5, 16, 2561),
    (5, 34, 64, 512), (5, 34, 64, 513)])
def test_adjoint_either_side_of_its_limits(rows, cols, C, B):
    """Outputs and gradients of sets at the ends of the batch against those of a few sets
    alone.  Both are float32 sweeps of the same steps: within 2e-5 of the largest
    gradient, the bound that the sweeps meet against complex128."""
    torch = _torch()
    from mentpy_amd.gradients.adjoint import AdjointEngine
    g, sim = _sim(rows, cols)
    eng = AdjointEngine(sim.simulator.plan)
    gen = torch.Generator().manual_seed(rows * cols)
    th = (torch.rand((B, len(g.trainable_nodes)), generator=gen) * 6.2).cuda()
    x = torch.randn((C, 1 << rows), generator=gen, dtype=torch.complex64).cuda()
    x = x / torch.linalg.vector_norm(x, dim=1, keepdim=True)
    seed = torch.randn((B, C, 1 << rows), generator=gen, dtype=torch.complex64).cuda() * 2.0 ** (-rows / 2)
    out, state = eng.forward(th, x)
    grad = eng.backward(state, seed)
    assert torch.isfinite(grad).all()
    for part in (slice(0, 3), slice(B - 3, B)):
        o, st = eng.forward(th[part].contiguous(), x)
        gr = eng.backward(st, seed[part].contiguous())
        assert (out[part] - o).abs().max().item() < 2e-5
        assert (grad[part] - gr).abs().max().item() < 2e-5 * max(1.0, gr.abs().max().item())


@pytest.mark.parametrize("sampled", [False, True])
def test_more_threads_than_one_launch_takes(sampled, rng):
    """14 slots take 1,024 threads per simulation: 4,194,304 simulations are 2^32 threads,
    more than one launch has.  The last ones (in the second launch) and those around
    the end of the first equal small launches; sampled, they meet their own draws."""
    torch = _torch()
    import mentpy_amd as mp
    g = mp.templates.linear_cluster(16)
    kw = {"force0": False, "seed": 4} if sampled else {}
    sim = mp.PatternSimulator(g, backend="hip-sv", window_size=15, **kw)
    assert sim.simulator.plan.info["n_slots"] == 14
    B = (1 << 22) + 3
    gen = torch.Generator(device="cuda").manual_seed(1)
    th = torch.rand((B, len(g.trainable_nodes)), generator=gen, device="cuda") * 6.2
    psi = haar_state(1, rng)
    out = sim.run_batch(th, psi)
    torch.cuda.synchronize()
    norm = torch.linalg.vector_norm(out, dim=-1)
    assert (norm - 1).abs().max().item() < 1e-5      # every row written
    post = mp.PatternSimulator(g, backend="hip-sv", window_size=15)
    for part in (slice(0, 2), slice((1 << 22) - 3, B)):
        want = post.run_batch(th[part].contiguous(), psi)
        if sampled:   # equal up to a global phase
            overlap = (want.conj() * out[part]).sum(-1).abs()
            assert (overlap - 1).abs().max().item() < 1e-5
        else:
            assert torch.equal(out[part], want)
