"""The fused TECE operator's copies of the weights (GPU)."""

import pytest
import torch

from tace_amd import model as pm
from tace_amd import ops, tece

pytestmark = pytest.mark.gpu


def _layer(cuda, dtype, mixing=None, C=32, H=2, A=16, n=20, E=300):
    """(forward of (x, R), conv, mlp, inputs) of one TECE convolution."""
    g = torch.Generator().manual_seed(5)
    torch.manual_seed(5)
    conv = tece.TeceConvolution(2, 2, C, H, A, 8)
    mlp = pm.MLP([8, 64, 64, conv.weight_numel])
    for m in (conv, mlp):
        m.to(dtype).to(cuda).requires_grad_(False)
    conv.mixing = mixing
    ei = torch.randint(0, n, (2, E), generator=g).to(cuda)
    vec = torch.randn(E, 3, generator=g, dtype=torch.float64).to(dtype).to(cuda)
    r = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).to(dtype).to(cuda).requires_grad_(True)
    x, R, W = r(n, 9 * C), r(E, 8), ops.edge_wigner(vec, 2).detach().requires_grad_(True)
    plan = ops.EdgePlan.from_edge_index(ei, n)
    nm = torch.arange(n, dtype=torch.int32, device=cuda)
    f = lambda chunk=10 ** 6: tece.tece_fused(conv, mlp, x, nm, R, plan, ei[0], ei[1], W, chunk)
    return f, conv, mlp, (x, R, W)


FORMS = [(torch.float64, None, True), (torch.float32, None, True), (torch.float32, None, False),
         (torch.float32, torch.bfloat16, True), (torch.float32, torch.bfloat16, False)]


@pytest.mark.parametrize("dtype,mixing,kernels", FORMS)
@pytest.mark.parametrize("strided", [False, True])
def test_backward_is_of_the_forwards_weights(cuda, dtype, mixing, kernels, strided, monkeypatch):
    """Weights written between forward and backward do not reach the backward
    of the forward before (all products on the kernels, on the library; weights
    that the kernels' layout does not take)."""
    monkeypatch.setattr(tece, "SO2_GEMM", kernels)
    monkeypatch.setattr(tece, "F32_GEMM", kernels)
    f, conv, mlp, inputs = _layer(cuda, dtype, mixing)
    if strided:
        w = conv.key_proj.m0_rlinear.weight
        w.data = w.data.t().contiguous().t()
    out = f()
    go = torch.randn(out.shape, generator=torch.Generator().manual_seed(1), dtype=torch.float64).to(out)
    want = torch.autograd.grad(out, inputs, go)
    again = f()
    lins = [m for m in mlp.mlp if hasattr(m, "alpha")]
    with torch.no_grad():
        for m in (conv.key_proj, conv.query_proj, conv.linear_down, conv.linear_coefs, conv.linear_glu, conv.linear_up,
                  conv.radial_proj, *lins[:-1]):
            for name, p in m.named_parameters():
                if name.endswith("weight"):
                    p.mul_(-1.5)
    got = torch.autograd.grad(again, inputs, go)
    assert torch.equal(out, again)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert not torch.equal(f(), out)
