"""Accuracy of the MB-QML products against 64 bits, with tolerances from the roundings that
their sums may have."""
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24   # half a unit in the last place of 1: the largest relative rounding


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def _chains(length, count):
    """Standard deviation, relative to the result, of `count` independent sums of `length`
    equal positive terms: an addition rounds its partial sum by U / sqrt(3), and the partial
    sums of n terms have a mean square of n^2 / 3."""
    return U / 3 * (length / count) ** 0.5


@pytest.mark.parametrize("B,K,S", [(16, 16, 8192), (5, 16, 32768), (33, 48, 20000)])
def test_long_contractions_in_partial_sums(B, K, S):
    """Seeds -2 / S sum_s f_s DC[s][k] over many inputs, all terms positive, f exact (t has
    one entry).  Sums of 64 terms (16 additions: a matrix instruction adds four), S / 64 of
    them; eight accumulators (two per wave) add S / 512 of those each; then the eight,
    and the scale.  One sum of S / 8 terms per accumulator has four times the additions
    per sum or more, in eight sums."""
    torch = _torch()
    from mentpy_amd import _native as nat
    L = nat.lib()
    gen = torch.Generator().manual_seed(S)
    DT = torch.zeros((K, S), dtype=torch.complex64)
    DT[0] = torch.rand(S, generator=gen) + 0.5
    DC = (torch.rand((S, K), generator=gen) + 0.5).to(torch.complex64)
    t = torch.zeros((B, K), dtype=torch.complex64)
    t[:, 0] = 2.0 ** torch.arange(B).remainder(3)
    want = -2.0 / S * torch.matmul(torch.matmul(t.to(torch.complex128), DT.to(torch.complex128)),
                                   DC.to(torch.complex128))
    t, DT, DC = t.cuda(), DT.cuda(), DC.cuda()
    seed = torch.full((B, K), complex("nan"), dtype=torch.complex64, device="cuda")
    ws = torch.empty(int(L.mbqc_transfer_workspace_bytes(B, S)), dtype=torch.uint8, device="cuda")
    nat.launch(t.device, L.mbqc_transfer_loss_seed_c64, t.data_ptr(), DT.data_ptr(), DC.data_ptr(), B, K,
               S, None, seed.data_ptr(), ws.data_ptr())
    got = seed.cpu().to(torch.complex128)
    # rows of t are multiples of one: K different sums
    rms = float(((got - want).real[0] / want.real[0]).pow(2).mean().sqrt())
    parts = [_chains(16, S / 64), _chains(S / 512, 8), _chains(8, 1), U / 3 ** 0.5]
    derived = sum(p * p for p in parts) ** 0.5
    print(f"{S} terms: relative rms error {rms:.2e}, derived {derived:.2e}", flush=True)
    assert torch.isfinite(seed).all() and rms < 2 * derived
