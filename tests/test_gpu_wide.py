"""Register-blocked statevector kernels of 7..20-slot windows: every window
size (its own split over lanes, registers and LDS exchanges), plans off the
grid's column structure, partly filled last workgroups, against the
complex128 oracle; compile-time and table step forms bit-identical."""
import numpy as np
import pytest

from conftest import haar_state

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


# (rows, cols, window, angle vectors, inputs): the default window is rows + 1;
# a wider one gives a plan with rows + 1 live slots whose steps are not a
# column's.  Batches leave a partly filled last workgroup where several
# simulations share one; 7x12 crosses a coefficient chunk and a rescale.
CASES = [(7, 12, None, 5, 3), (8, 4, None, 3, 1), (9, 5, None, 1, 1), (9, 4, None, 7, 2),
         (10, 3, None, 2, 1), (11, 3, None, 1, 2), (12, 3, None, 1, 1), (13, 3, None, 1, 1),
         (14, 3, None, 1, 1), (15, 3, None, 2, 1), (16, 3, None, 1, 2), (17, 3, None, 1, 1), (19, 3, None, 1, 1),
         (6, 5, 8, 5, 1), (7, 4, 9, 3, 3), (8, 4, 10, 2, 1), (9, 3, 11, 1, 2), (14, 3, 16, 1, 1),
         (15, 3, 17, 1, 1)]


@pytest.mark.parametrize("rows,cols,window,B,S", CASES)
def test_wide_windows_match_oracle(rows, cols, window, B, S, rng):
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.simulators.hip_simulator import sv_forward, _as_angles, _as_states
    from oracle.vectorized import sv_batch
    g = mp.templates.grid_cluster(rows, cols)
    sim = mp.PatternSimulator(g, backend="hip-sv", **({"window_size": window} if window else {}))
    plan = sim.simulator.plan
    assert plan.info["n_slots"] == (window - 1 if window else rows)
    th = rng.uniform(-7, 7, (B, len(g.trainable_nodes))).astype(np.float32)
    psi = np.stack([haar_state(rows, rng) for _ in range(S)])
    dev = torch.device("cuda")
    a, s = _as_angles(th, plan.info["n_angles"], dev), _as_states(psi, plan.info["n_inputs"], dev)
    guard = torch.full((B + 1, S, 1 << rows), 7.0, dtype=torch.complex64, device=dev)
    out = sv_forward(plan, a, s, out=guard[:B])
    table = sv_forward(plan, a, s, table_steps=True)
    torch.cuda.synchronize()
    assert torch.equal(out, table), "compile-time and table steps differ"
    assert (guard[B] == 7.0).all(), "a store past the last simulation"
    ref = sv_batch(g, th.astype(np.float64), psi)
    err = np.abs(out.cpu().numpy() - ref).max()
    # complex64 butterflies: each step adds about one rounding (6e-8) to amplitudes below 1
    assert err < 2e-5, f"amplitude error {err}"


def _grid_outputs(a, x, rows, cols):
    """Raw-phase outputs of a grid pattern, differentiable in complex128: angles
    a [B, n], inputs x [C, 2^rows]."""
    torch = _torch()
    B, C, d = a.shape[0], x.shape[0], 1 << rows
    j = torch.arange(d, device="cuda")
    bit = [((j >> (rows - 1 - i)) & 1).double() for i in range(rows)]
    t = x.to(torch.complex128)
    for i in range(rows - 1):
        t = t * (1 - 2 * bit[i] * bit[i + 1])
    t = t[None].expand(B, -1, -1)
    for k in range(rows * (cols - 1)):
        i, col = k % rows, k // rows
        ph = torch.polar(torch.ones_like(a[:, 0]), -a[:, i * (cols - 1) + col])
        v = t.reshape(B, C, 1 << i, 2, -1)
        p, q = v[:, :, :, 0], v[:, :, :, 1] * ph[:, None, None, None]
        t = (torch.stack([p + q, p - q], 3) * 0.5 ** 0.5).reshape(B, C, d)
        if i:
            t = t * (1 - 2 * bit[i - 1] * bit[i])
    return t


@pytest.mark.parametrize("rows,cols,C,B", [(6, 14, 4, 5), (6, 14, 128, 512), (7, 12, 3, 2), (8, 4, 16, 3),
                                           (9, 4, 1, 3), (10, 4, 2, 1), (11, 3, 4, 1), (12, 3, 2, 1),
                                           (13, 3, 2, 1), (14, 3, 1, 1),
                                           (4, 5, 1, 1), (4, 20, 16, 5), (4, 19, 12, 3), (4, 6, 128, 3),
                                           (4, 5, 16, 2048), (4, 5, 16, 2049), (5, 4, 1, 1),
                                           (5, 15, 32, 7), (5, 16, 3, 2), (5, 5, 24, 2048),
                                           (5, 5, 24, 2049)])
def test_wide_adjoint_matches_complex128(rows, cols, C, B, rng):
    """Outputs and angle gradients of the register-blocked adjoint sweeps
    against torch autograd on the complex128 grid steps: one and several
    simulations per wave and per row, rows of 64 columns, checkpoint pairs
    (65,536 columns), a rescale (more than 64 steps), shared and unshared
    coefficients, the last and the first column count on either side of the
    4- and 5-slot limits."""
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.gradients.adjoint import pattern_sv
    g = mp.templates.grid_cluster(rows, cols)
    sim = mp.PatternSimulator(g, backend="hip-sv")
    n, d = len(g.trainable_nodes), 1 << rows
    gen = torch.Generator().manual_seed(rows)
    th = (torch.rand((B, n), generator=gen) * 6.2).cuda().requires_grad_(True)
    x = torch.randn((C, d), generator=gen, dtype=torch.complex64).cuda()
    x = x / torch.linalg.vector_norm(x, dim=1, keepdim=True)
    cot = torch.randn((B, C, d), generator=gen, dtype=torch.complex64).cuda() / d ** 0.5
    out = pattern_sv(sim, th, x)
    grad, = torch.autograd.grad(out, th, cot)
    bs = list(range(B)) if B < 8 else [0, B // 2, B - 1]
    a = th.detach()[bs].double().requires_grad_(True)
    t = _grid_outputs(a, x, rows, cols)
    want, = torch.autograd.grad(t, a, cot[bs].to(torch.complex128))
    oerr = (out.detach()[bs] - t.detach()).abs().max().item()
    scale = want.abs().max().item()
    gerr = (grad[bs] - want).abs().max().item()
    # one rounding (6e-8) per step on unit-norm states and cotangents of norm about
    # sqrt(2 C): far below 2e-5 of the largest entry
    assert oerr < 2e-5, f"output error {oerr}"
    assert gerr < 2e-5 * max(scale, 1.0), f"gradient error {gerr} of {scale}"


@pytest.mark.parametrize("rows,cols,C,B", [(2, 4, 4, 1), (2, 34, 4, 67), (3, 5, 3, 4), (3, 24, 8, 5),
                                           (4, 3, 16, 1), (4, 18, 16, 6), (4, 6, 17, 2048),
                                           (4, 6, 1, 2049), (4, 18, 16, 2051), (5, 4, 32, 1),
                                           (5, 14, 33, 3)])
def test_gradient_from_outputs_matches_complex128(rows, cols, C, B, rng):
    """Angle gradients from outputs and cotangents alone against torch autograd on
    the complex128 grid steps: every window, one and two register digits on
    either side of their limit, partly filled last workgroups, several
    coefficient chunks, fewer, as many and more columns than the transfer matrix."""
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd import _native as nat
    g = mp.templates.grid_cluster(rows, cols)
    sim = mp.PatternSimulator(g, backend="hip-sv")
    plan = sim.simulator.plan
    assert nat.lib().mbqc_sv_has_outputs_gradient(plan.handle) == 1
    n, d = len(g.trainable_nodes), 1 << rows
    gen = torch.Generator().manual_seed(rows * cols)
    th = (torch.rand((B, n), generator=gen) * 6.2).cuda()
    x = torch.randn((C, d), generator=gen, dtype=torch.complex64).cuda()
    x = x / torch.linalg.vector_norm(x, dim=1, keepdim=True)
    cot = torch.randn((B, C, d), generator=gen, dtype=torch.complex64).cuda() / d ** 0.5
    bs = list(range(B)) if B < 8 else [0, B // 2, B - 1]
    a = th[bs].double().requires_grad_(True)
    t = _grid_outputs(a, x, rows, cols)
    want, = torch.autograd.grad(t, a, cot[bs].to(torch.complex128))
    out = torch.empty((B, C, d), dtype=torch.complex64, device="cuda")
    grad = torch.full((B, n), float("nan"), device="cuda")
    loss = torch.full((B,), float("nan"), device="cuda")
    nat.launch(out.device, nat.lib().mbqc_sv_forward_c64, plan.handle, th.data_ptr(), n, 1,
               x.data_ptr(), d, out.data_ptr(), None, B, C, 0)
    nat.launch(out.device, nat.lib().mbqc_sv_outputs_gradient_c64, plan.handle, th.data_ptr(), n, 1,
               out.data_ptr(), cot.data_ptr(), B, C, loss.data_ptr(), grad.data_ptr())
    assert torch.isfinite(grad).all()
    # one rounding (6e-8) per step on coefficients of norm about sqrt(2 C): far
    # below 2e-5 of the largest entry
    gerr = (grad[bs] - want).abs().max().item()
    scale = want.abs().max().item()
    assert gerr < 2e-5 * max(scale, 1.0), f"gradient error {gerr} of {scale}"
    wl = 1 + 0.5 * (t.detach() * cot[bs].to(torch.complex128).conj()).real.sum((1, 2))
    assert (loss[bs] - wl).abs().max().item() < 2e-5 * C ** 0.5


@pytest.mark.parametrize("B,K,S", [(1, 16, 1), (15, 20, 16), (17, 64, 33), (33, 1024, 100), (2049, 256, 37),
                                   (1030, 1024, 65), (16400, 64, 257), (4097, 256, 256),
                                   (1031, 256, 257), (4097, 64, 100)])
def test_transfer_products_match_complex128(B, K, S, rng):
    """Loss and seed through the data matrix, every tiling: partly filled tiles of
    rows and columns, a contraction length with a remainder, loss alone and
    seed alone; the Gram seed of the same data."""
    torch = _torch()
    from mentpy_amd import _native as nat
    L = nat.lib()
    gen = torch.Generator().manual_seed(B + K + S)
    t = torch.randn((B, K), generator=gen, dtype=torch.complex64).cuda() / K ** 0.5
    D = torch.randn((S, K), generator=gen, dtype=torch.complex64).cuda()
    DT, DC = D.t().contiguous(), D.conj().resolve_conj().contiguous()
    ws = torch.empty(int(L.mbqc_transfer_workspace_bytes(B, S)), dtype=torch.uint8, device="cuda")
    dev = t.device

    def both(loss, seed):
        nat.launch(dev, L.mbqc_transfer_loss_seed_c64, t.data_ptr(), DT.data_ptr(), DC.data_ptr(), B, K, S,
                   loss, seed, ws.data_ptr())
    l0, l1 = (torch.full((B,), float("nan"), device="cuda") for _ in range(2))
    s0, s1, s2 = (torch.full((B, K), float("nan"), dtype=torch.complex64, device="cuda") for _ in range(3))
    both(l0.data_ptr(), s0.data_ptr())
    both(l1.data_ptr(), None)
    both(None, s1.data_ptr())
    assert torch.equal(l0, l1) and torch.equal(s0, s1)
    MT = (D.to(torch.complex128).conj().t() @ D.to(torch.complex128)).t().to(torch.complex64).contiguous()
    nat.launch(dev, L.mbqc_gram_seed_c64, t.data_ptr(), MT.data_ptr(), B, K, S, s2.data_ptr())
    f = t.to(torch.complex128) @ D.to(torch.complex128).t()
    want_loss = 1 - (f.abs() ** 2).mean(1)
    want = -2.0 / S * (f @ D.to(torch.complex128).conj())
    # sums of K (S) products of size 1/K (1) and one rounding (6e-8) each
    assert (l0 - want_loss).abs().max().item() < 1e-5 * want_loss.abs().max().item()
    for s in (s0, s2):
        assert (s - want).abs().max().item() < 1e-5 * want.abs().max().item()


def test_gradient_from_outputs_refuses_other_plans():
    """Six rows, and a window with spare slots."""
    _torch()
    import mentpy_amd as mp
    from mentpy_amd import _native as nat
    for rows, kw in ((6, {}), (3, {"window_size": 5})):
        sim = mp.PatternSimulator(mp.templates.grid_cluster(rows, 4), backend="hip-sv", **kw)
        assert nat.lib().mbqc_sv_has_outputs_gradient(sim.simulator.plan.handle) == 0


@pytest.mark.parametrize("rows,cols,window,B,S", [
    (2, 5, None, 1, 1), (2, 40, None, 2050, 1), (3, 5, None, 1, 1), (3, 30, None, 7, 3),
    (4, 20, None, 1, 1), (4, 20, None, 1023, 2), (4, 5, None, 4, 4096), (5, 14, None, 9, 1),
    (5, 6, None, 2049, 1), (6, 13, None, 3, 1), (6, 5, None, 1100, 3), (3, 6, 5, 5, 3),
    (4, 6, 6, 5, 300), (5, 5, 7, 11, 1), (2, 6, 7, 3, 2)])
def test_narrow_windows_small_batches(rows, cols, window, B, S, rng):
    """Batches below the one-simulation-per-lane kernel's share of the chip: a
    whole wave or a few lanes per simulation, partly filled last workgroups,
    several coefficient chunks, column and general plans."""
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.simulators.hip_simulator import sv_forward, _as_angles, _as_states
    from oracle.vectorized import sv_batch
    g = mp.templates.grid_cluster(rows, cols)
    sim = mp.PatternSimulator(g, backend="hip-sv", **({"window_size": window} if window else {}))
    plan = sim.simulator.plan
    th = rng.uniform(-7, 7, (B, len(g.trainable_nodes))).astype(np.float32)
    psi = np.stack([haar_state(rows, rng) for _ in range(S)])
    dev = torch.device("cuda")
    a, s = _as_angles(th, plan.info["n_angles"], dev), _as_states(psi, plan.info["n_inputs"], dev)
    guard = torch.full((B + 1, S, 1 << rows), 7.0, dtype=torch.complex64, device=dev)
    out, phase = sv_forward(plan, a, s, out=guard[:B], want_phase=True)
    table = sv_forward(plan, a, s, table_steps=True)
    raw = sv_forward(plan, a, s, ref_phase=False, renormalize=False)
    torch.cuda.synchronize()
    assert torch.equal(out, table), "compile-time and table steps differ"
    assert (guard[B] == 7.0).all(), "a store past the last simulation"
    rows_b = sorted({0, B // 2, B - 1})
    ref = sv_batch(g, th[rows_b].astype(np.float64), psi)
    assert np.abs(out[rows_b].cpu().numpy() - ref).max() < 2e-5
    assert (raw * phase[..., None] - out).abs().max().item() < 2e-5


@pytest.mark.parametrize("rows,cols,window,B,S", [
    (4, 5, None, 257, 4), (4, 19, None, 129, 16), (4, 7, None, 2731, 12), (4, 7, None, 2732, 12),
    (5, 16, None, 100, 32), (5, 6, None, 8193, 4), (6, 13, None, 41, 64), (6, 5, None, 32769, 4),
    (4, 6, 7, 300, 8)])
def test_shared_coefficients_equal_single_inputs(rows, cols, window, B, S, rng):
    """Raw-phase launches whose inputs share their angles' coefficients (4, 8, 16
    and more in a row, either side of the largest batches, general plans) equal
    the launches of one input each bit for bit."""
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.simulators.hip_simulator import sv_forward
    g = mp.templates.grid_cluster(rows, cols)
    sim = mp.PatternSimulator(g, backend="hip-sv", **({"window_size": window} if window else {}))
    plan = sim.simulator.plan
    gen = torch.Generator().manual_seed(rows * cols)
    th = (torch.rand((B, len(g.trainable_nodes)), generator=gen) * 12 - 6).cuda()
    x = torch.randn((S, 1 << rows), generator=gen, dtype=torch.complex64).cuda()
    for renorm in (False, True):
        got = sv_forward(plan, th, x, ref_phase=False, renormalize=renorm)
        for i in range(0, S, max(1, S // 4)):
            one = sv_forward(plan, th, x[i:i + 1], ref_phase=False, renormalize=renorm)
            assert torch.equal(got[:, i], one[:, 0])


@pytest.mark.parametrize("rows,B", [(2, 4097), (3, 2049), (4, 16385), (5, 16385), (6, 32769)])
def test_narrow_windows_lane_kernel_above_the_threshold(rows, B, rng):
    """The first batch above the threshold (one simulation per lane) against
    the oracle and, row by row, against the small-batch kernel."""
    torch = _torch()
    import mentpy_amd as mp
    from oracle.vectorized import sv_batch
    g = mp.templates.grid_cluster(rows, 9)
    sim = mp.PatternSimulator(g, backend="hip-sv")
    gen = torch.Generator().manual_seed(rows)
    th = (torch.rand((B, len(g.trainable_nodes)), generator=gen) * 6.2).cuda()
    psi = haar_state(rows, rng)
    full = sim.run_batch(th, psi)
    small = sim.run_batch(th[-40:].contiguous(), psi)
    assert torch.equal(full[-40:], small), "the two kernels differ"
    ref = sv_batch(g, th[:8].double().cpu().numpy(), psi[None])
    assert np.abs(full[:8].cpu().numpy() - ref).max() < 2e-5


@pytest.mark.parametrize("rows,cols,window", [(1, 7, None), (2, 5, None), (3, 4, 5), (4, 20, None),
                                              (5, 14, None), (6, 30, None), (4, 6, 7)])
def test_host_runs_equal_batched_runs(rows, cols, window, rng):
    """run() as one native call on host memory against run_batch on device
    tensors, bit for bit; raw phase and no renormalisation too; calls from
    several threads and on a side stream."""
    import threading
    torch = _torch()
    import mentpy_amd as mp
    g = mp.templates.linear_cluster(cols) if rows == 1 else mp.templates.grid_cluster(rows, cols)
    n = len(g.trainable_nodes)
    psi = [haar_state(rows, rng) for _ in range(3)]
    th = rng.uniform(-7, 7, (3, n))
    kw = {"window_size": window} if window else {}
    for extra in ({}, {"phase": "raw"}, {"renormalize": False}):
        sim = mp.PatternSimulator(g, backend="hip-sv", **kw, **extra)
        assert sim.simulator._host_run
        for t, x in zip(th, psi):
            sim.reset(x)
            got = sim.run(t, output_form="sv")
            want = sim.run_batch(t, x)[0, 0].cpu().numpy().astype(np.complex128)
            assert got.dtype == np.complex128 and np.array_equal(got, want)
    want = [sim.run_batch(t, x)[0, 0].cpu().numpy() for t, x in zip(th, psi)]
    bad = []

    def work(i):
        s = mp.PatternSimulator(g, backend="hip-sv", renormalize=False, **kw)
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(50):
                s.reset(psi[i])
                if not np.array_equal(s.run(th[i], output_form="sv"), want[i]):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("waves,wg_waves,max_rows", [(1, 1, 5), (4, 4, 6), (33, 3, 5), (4096, 4, 6)])
def test_batched_register_groups_in_one_launch(waves, wg_waves, max_rows, rng):
    """Every register group of a batch in one kernel, its items dealt to lists:
    fewer waves than lists, a ragged last workgroup, more waves than items; the
    outputs equal the launch with a kernel per group bit for bit."""
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.batched import BatchedForward
    jobs = []
    for i in range(23):
        r = 1 + i % max_rows
        g = mp.templates.linear_cluster(5 + i) if r == 1 else mp.templates.grid_cluster(r, 4 + i % 7)
        sim = mp.PatternSimulator(g, backend="hip-sv")
        S = (16, 3, 1)[i % 3]
        th = rng.uniform(0, 6, (7 + 11 * i, len(g.trainable_nodes))).astype(np.float32)
        jobs.append((sim, th, np.stack([haar_state(r, rng) for _ in range(S)])))
    bf = BatchedForward(jobs)
    sizes = [64 if ns in bf.groups() else 0 for ns in range(max_rows + 1)]
    want = [o.clone() for o in bf.launch(wg_waves=1, group_waves=sizes)]
    for _ in range(2):
        for o in bf.outputs:
            o.zero_()
        got = bf.launch(waves=max(waves, wg_waves), wg_waves=wg_waves)
        torch.cuda.synchronize()
        for x, y in zip(got, want):
            assert torch.equal(x, y)
    for (sim, th, st), o in zip(jobs, want):
        assert (sim.run_batch(th, st) - o).abs().max().item() < 1e-6


@pytest.mark.parametrize("rows,cols,window,B,S", [
    (2, 4, None, 1, 1), (2, 30, None, 37, 3), (3, 12, None, 130, 1), (3, 4, None, 1, 2),
    (4, 6, None, 9, 2), (4, 5, None, 2049, 1), (5, 6, None, 5, 1), (6, 4, None, 3, 1),
    (7, 3, None, 2, 1), (2, 5, 4, 17, 2), (2, 5, 5, 9, 1), (3, 4, 5, 9, 1), (3, 5, 6, 3, 2),
    (4, 4, 6, 5, 1), (4, 5, 7, 3, 1), (5, 4, 8, 2, 1), (1, 6, 3, 50, 2)])
def test_density_matrices_of_column_and_other_plans(rows, cols, window, B, S, rng):
    """Pauli-vector kernels of column plans (one and two register digits, more
    steps than a coefficient chunk) and the matrix kernels of the other plans
    (a window above the grid's own), with and without noise and trace
    normalisation, against the oracle; nothing stored past the last matrix."""
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.noise import NoiseModel
    from mentpy_amd.simulators.hip_simulator import dm_forward, _as_angles, _as_states
    from oracle.vectorized import dm_batch
    g = mp.templates.linear_cluster(cols) if rows == 1 else mp.templates.grid_cluster(rows, cols)
    sim = mp.PatternSimulator(g, backend="hip-dm", **({"window_size": window} if window else {}))
    plan = sim.simulator.plan
    th = rng.uniform(-7, 7, (B, len(g.trainable_nodes))).astype(np.float32)
    psi = np.stack([haar_state(rows, rng) for _ in range(S)])
    dev = torch.device("cuda")
    a, s = _as_angles(th, plan.info["n_angles"], dev), _as_states(psi, plan.info["n_inputs"], dev)
    d = 1 << rows
    at = sorted({0, B // 2, B - 1})
    for pd, pr in ((0.0, 0.0), (0.03, 0.01)):
        guard = torch.full((B + 1, S, d, d), 7.0, dtype=torch.complex64, device=dev)
        out = dm_forward(plan, a, s, p_depol=pd, p_readout=pr, out=guard[:B])
        raw = dm_forward(plan, a, s, p_depol=pd, p_readout=pr, renormalize=False)
        torch.cuda.synchronize()
        assert (guard[B] == 7.0).all()
        ref = dm_batch(g, th[at].astype(np.float64), psi, p_depol=pd, p_readout=pr)
        assert np.abs(out[at].cpu().numpy() - ref).max() < 2e-5
        assert (raw - out).abs().max().item() < 2e-5
    if window is None:   # the damping channels' population shift on the outputs
        noise = NoiseModel(amplitude_damping=0.2, gad_gamma=0.1, gad_p=0.7, phase_flip=0.05)
        got = dm_forward(plan, a, s, noise=noise)
        gen = dm_forward(plan, a, s, noise=noise, step_probs=True)
        assert (got - gen).abs().max().item() < 2e-5


@pytest.mark.parametrize("rows,cols,B,pad", [(4, 19, 131073, 0), (4, 19, 131071, 0), (3, 25, 131073, 5),
                                             (6, 40, 40331, 0), (5, 40, 65536, 1)])
def test_row_major_angles_equal_angle_major(rows, cols, B, pad, rng):
    """Large batches of row-major angles (on either side of the copy's byte limit,
    odd batches, padded rows) against angle-major ones, run and sampled, bit for
    bit, and inside a captured graph."""
    torch = _torch()
    import mentpy_amd as mp
    g = mp.templates.grid_cluster(rows, cols)
    n = len(g.trainable_nodes)
    sim = mp.PatternSimulator(g, backend="hip-sv")
    gen = torch.Generator(device="cuda").manual_seed(rows)
    a = torch.rand((B, n + pad), generator=gen, device="cuda")[:, :n]
    am = a.t().contiguous().t()
    psi = haar_state(rows, rng)
    want = sim.run_batch(am, psi)
    assert torch.equal(sim.run_batch(a, psi), want)
    out = [mp.PatternSimulator(g, backend="hip-sv", force0=False, seed=3).run_batch(x, psi) for x in (a, am)]
    assert torch.equal(out[0], out[1])
    x = torch.as_tensor(psi, device="cuda").to(torch.complex64)
    sim.run_batch(a, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = sim.run_batch(a, x)
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
