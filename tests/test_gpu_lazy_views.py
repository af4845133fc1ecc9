"""Lazily conjugated and negated tensors (torch's conj and neg views share the memory of the
tensor that they are taken from) as inputs, angles and cotangents."""
import numpy as np
import pytest

from conftest import haar_state

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


@pytest.mark.parametrize("rows", [3, 8])
def test_lazy_views_equal_their_values(rows, rng):
    torch = _torch()
    import mentpy_amd as mp
    from mentpy_amd.gradients.adjoint import pattern_sv
    g = mp.templates.grid_cluster(rows, 4)
    n = len(g.trainable_nodes)
    sim = mp.PatternSimulator(g, backend="hip-sv")
    x = torch.as_tensor(np.stack([haar_state(rows, rng) for _ in range(3)]), dtype=torch.complex64,
                        device="cuda").conj()
    z = torch.randn((5, n), dtype=torch.complex64, device="cuda").conj().imag
    assert x.is_conj() and z.is_neg()
    want = sim.run_batch(z.resolve_neg().clone(), x.resolve_conj().clone())
    assert torch.equal(sim.run_batch(z, x), want)
    # the cotangent of a conjugated output is a conjugated view
    y = torch.randn((5, 3, 1 << rows), dtype=torch.complex64, device="cuda")
    a = z.resolve_neg().clone().requires_grad_(True)

    def loss(conj):
        out = pattern_sv(sim, a, x)
        return (conj(out) * y).sum().real

    got, = torch.autograd.grad(loss(torch.conj), a)
    ref, = torch.autograd.grad(loss(lambda v: torch.complex(v.real, -v.imag)), a)
    assert torch.equal(got, ref)
