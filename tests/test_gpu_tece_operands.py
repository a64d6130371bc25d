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


def _params(conv, mlp):
    P = tece._FusedParams(conv, mlp, torch.float32)
    return P, [o.frag for T in (P.k_T, P.k_N, P.q_T, P.q_N, P.d_T, P.d_N, P.s_T, P.s_N) for o in T] + [
        P.s_b, P.mlp_flat, P.rp_T, P.rp_N]


def test_nothing_is_kept_and_scales_are_read(cuda):
    """Another scale of a linear makes other operands; a call leaves nothing on the module."""
    f, conv, mlp, _ = _layer(cuda, torch.float32)
    before = set(vars(conv))
    out = f()
    conv.linear_down.m0_rlinear.alpha *= 2
    twice = f()
    conv.linear_down.m0_rlinear.alpha /= 2
    assert set(vars(conv)) == before
    assert not torch.equal(twice, out) and torch.equal(f(), out)


@pytest.mark.parametrize("mixing", [None, torch.bfloat16])
def test_operands_in_a_recorded_graph(cuda, mixing):
    """The layout recorded at its first call; replays read the weights as they
    are then, also after the module has moved to other weights and been used."""
    f, conv, mlp, _ = _layer(cuda, torch.float32, mixing)
    held = [p.data for m in (conv, mlp) for p in m.parameters()]   # the recorded weights stay
    graph = torch.cuda.CUDAGraph()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        conv.temperature_logit.sigmoid()
    torch.cuda.current_stream().wait_stream(s)
    with torch.cuda.graph(graph):
        P, got = _params(conv, mlp)
    eager = lambda: [t.clone() for t in _params(conv, mlp)[1]]
    for step in range(3):
        with torch.no_grad():
            for p in held:
                p.mul_(1.25)
        want = eager()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, want)), step
    for m in (conv, mlp):   # other storages; the graph keeps to the recorded ones
        for p in m.parameters():
            p.data = p.data.clone().mul_(3.0)
    f()
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(got, want))
