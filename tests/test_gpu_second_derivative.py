"""Kernels with a first derivative only refuse a second one, wherever it is asked for (GPU)."""

import pytest
import torch

from tace_amd import model as pm
from tace_amd import ops
from tace_amd.so3 import Irrep, Irreps

pytestmark = pytest.mark.gpu


def _gate(L, C, n, cuda):
    """(gate function of x, x) of the kernel's layout (L = 4: more blocks than it takes)."""
    irr = [(C, Irrep(l, (-1) ** l)) for l in range(L + 1)]
    lout = pm.GMLayout(Irreps(irr))
    lin = pm.GMLayout(Irreps([((L + 2) * C, Irrep(0, 1))] + irr[1:]))
    assert pm._GateFn.native(lin, lout, C) == (L < 4)
    x = torch.randn(n, lin.dim, generator=torch.Generator().manual_seed(L)).to(cuda).requires_grad_(True)
    return lambda v: pm._gate(v, lin, lout, C), x


@pytest.mark.parametrize("L", [0, 3, 4])
def test_gate(cuda, L):
    """Outside ``ops.differentiable_twice`` an error, inside it the derivative."""
    f, x = _gate(L, 8, 5, cuda)
    (first,) = torch.autograd.grad(f(x).square().sum(), x)
    with pytest.raises(RuntimeError, match="second derivative|out="):
        torch.autograd.grad(f(x).square().sum(), x, create_graph=True)
    with ops.differentiable_twice():
        (gx,) = torch.autograd.grad(f(x).square().sum(), x, create_graph=True)
        (second,) = torch.autograd.grad(gx.square().sum(), x)
    assert (gx - first).abs().max() < 1e-5 * first.abs().max()
    assert second.abs().max() > 0


def test_energy_head(cuda):
    n, C = 6, 32
    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g).to(cuda)
    i = lambda *v: torch.tensor(v, device=cuda)
    x = r(n, C).requires_grad_(True)
    E, en = ops.EnergyHead.apply(x, torch.arange(n, device=cuda), r(C, 16), r(16), r(n, 2), r(2), r(2), r(2),
                                 i(0, 0, 0, 0, 1, 1), i(0, 4, 6), torch.arange(n + 1, dtype=torch.int32, device=cuda))
    for out in (E, en):
        with pytest.raises(RuntimeError, match="second derivative"):
            torch.autograd.grad(out.sum(), x, create_graph=True, retain_graph=True)
    assert torch.autograd.grad(E.sum(), x)[0].shape == x.shape
