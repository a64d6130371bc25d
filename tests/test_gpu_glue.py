"""The gate, the energy readout, the edge-vector gradient and the key grouping kernels (GPU)."""

import pytest
import torch

from tace_amd import model as pm
from tace_amd import ops
from tace_amd.so3 import Irrep, Irreps

pytestmark = pytest.mark.gpu

# a handful of roundings per output (exp to 1 ulp, products, sums of at most 7 terms)
EPS = {torch.float32: 2e-6, torch.float64: 4e-15}


def _rel(got, want):
    return ((got.double() - want).abs().max() / want.abs().max().clamp_min(1e-300)).item()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("L,C,n,off", [(0, 64, 5, 0), (1, 5, 257, 0), (2, 128, 1, 0), (3, 128, 70, 0), (3, 33, 19, 0),
                                       (3, 64, 31, 1), (2, 256, 0, 0)])
def test_gate_matches_torch(cuda, dtype, L, C, n, off):
    """Gate kernels against the same expressions in float64: channel counts
    off the vector width, a misaligned input (off), no nodes."""
    lout = pm.GMLayout(Irreps([(C, Irrep(l, (-1) ** l)) for l in range(L + 1)]))
    lin = pm.GMLayout(Irreps([((L + 2) * C, Irrep(0, 1))] + [(C, Irrep(l, (-1) ** l)) for l in range(1, L + 1)]))
    assert pm._GateFn.native(lin, lout, C)
    g = torch.Generator().manual_seed(n + L)
    x64 = 3 * torch.randn(n, lin.dim, generator=g, dtype=torch.float64)
    go64 = torch.randn(n, lout.dim, generator=g, dtype=torch.float64)
    buf = torch.empty(n * lin.dim + off, dtype=dtype, device=cuda)
    x = buf[off:].view(n, lin.dim).copy_(x64).requires_grad_(True)
    go = go64.to(dtype).to(cuda)
    out = pm._GateFn.apply(x, lin, lout, C)
    (gx,) = torch.autograd.grad(out, x, go)
    assert out.shape == (n, lout.dim) and gx.shape == x.shape
    if n == 0:
        return
    xr = x.detach().double().cpu().requires_grad_(True)
    gate = torch.sigmoid(lin.block(xr, 0).view(n, -1)[:, :(L + 1) * C]) * pm.SIGMOID_CST
    want = torch.cat([(s * gate[:, k * C:(k + 1) * C].unsqueeze(1)).reshape(-1)
                      for k, s in enumerate(pm._gated_blocks(xr, lin, lout, C))]).view(n, -1)
    (gw,) = torch.autograd.grad(want, xr, go.double().cpu())
    assert _rel(out.detach().cpu(), want.detach()) < EPS[dtype]
    assert _rel(gx.cpu(), gw) < EPS[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("C,S,sizes", [(64, 1, [1]), (128, 4, [1, 30, 1]), (200, 89, [5, 64, 65, 1, 0, 700]),
                                       (512, 2, [3000]), (40, 70, [2, 2])])
def test_energy_head_matches_torch(cuda, dtype, C, S, sizes):
    """Readout, element tables and graph sums against float64: atoms alone
    with and without edges, an empty graph, more species than lanes."""
    g = torch.Generator().manual_seed(C)
    n = sum(sizes)
    mk = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).to(dtype)
    x, w1, w2, e0, sc, sh = mk(n, C), mk(C, 16) / C ** 0.5, mk(16), mk(S), mk(S), mk(S)
    attrs = torch.nn.functional.one_hot(torch.randint(0, S, (n,), generator=g), S).to(dtype)
    row_of = torch.randperm(n, generator=g)
    batch = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes))
    ptr = torch.tensor([0] + sizes).cumsum(0)
    deg = torch.randint(0, 3, (n,), generator=g)
    rowptr = torch.cat([torch.zeros(1, dtype=torch.int64), deg.cumsum(0)]).to(torch.int32)
    gE, gn = mk(len(sizes)), mk(n)
    d = lambda t: t.to(cuda)
    xg = d(x).requires_grad_(True)
    E, en = ops.EnergyHead.apply(xg, d(row_of), d(w1), d(w2), d(attrs), d(e0), d(sc), d(sh), d(batch), d(ptr), d(rowptr))
    got = torch.autograd.grad([E, en], xg, [d(gE), d(gn)], retain_graph=True)[0]
    only_e = torch.autograd.grad(E, xg, d(gE), retain_graph=True)[0]
    only_n = torch.autograd.grad(en, xg, d(gn))[0]
    xr = x.double().requires_grad_(True)
    e = torch.nn.functional.silu(xr[row_of] @ w1.double()) @ w2.double()
    keep = 1.0 - ((ptr[1:] - ptr[:-1])[batch] == 1).double() * (deg == 0).double()
    a = attrs.double()
    en_w = a @ e0.double() + (e * (a @ sc.double()) + a @ sh.double()) * keep
    E_w = torch.zeros(len(sizes), dtype=torch.float64).index_add(0, batch, en_w)
    want = torch.autograd.grad([E_w, en_w], xr, [gE.double(), gn.double()], retain_graph=True)[0]
    # sums of C products and of 16 hidden values in another order; the graphs'
    # energies of their nodes too, of whose magnitudes the rounding is a share
    tol = (C + 16) ** 0.5 * EPS[dtype]
    size = torch.zeros(len(sizes), dtype=torch.float64).index_add(0, batch, en_w.detach().abs())
    assert (E.detach().cpu().double() - E_w.detach()).abs().max() < tol * size.max()
    assert _rel(en.detach().cpu(), en_w.detach()) < tol
    assert _rel(got.cpu(), want) < tol
    assert _rel((only_e + only_n).cpu(), want) < tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("sorted_edges", [True, False])
def test_edge_vector_gradient_with_lattices(cuda, dtype, sorted_edges):
    """Position and lattice gradients of edge_vectors with ``ptr`` against
    autograd: nodes without edges, with 1, 15, 16, 17 and 100, a graph
    without edges."""
    g = torch.Generator().manual_seed(1)
    sizes = [7, 1, 130, 2]
    n = sum(sizes)
    ptr = torch.tensor([0] + sizes).cumsum(0)
    batch = torch.repeat_interleave(torch.arange(4), torch.tensor(sizes))
    src, dst = [], []
    for i, k in enumerate([0, 1, 15, 16, 17, 100] + [0] * (n - 6)):
        lo, hi = (0, 7) if i < 7 else (8, 138)
        if i >= 8 and i < 138:
            k = i % 20
        src.append(torch.randint(lo, hi, (k,), generator=g))
        dst.append(torch.full((k,), i))
    ei = torch.stack([torch.cat(src), torch.cat(dst)])
    if not sorted_edges:
        ei = ei[:, torch.randperm(ei.shape[1], generator=g)]
    E = ei.shape[1]
    pos, lat = torch.randn(n, 3, generator=g, dtype=dtype), torch.randn(4, 3, 3, generator=g, dtype=dtype)
    sh = torch.randint(-2, 3, (E, 3), generator=g).to(dtype)
    go = torch.randn(E, 3, generator=g, dtype=dtype)
    plan = ops.EdgePlan.from_edge_index(ei.to(cuda), n)
    assert (plan.eid is None) == sorted_edges
    p, l = pos.to(cuda).requires_grad_(True), lat.to(cuda).requires_grad_(True)
    eg = batch[ei[0]].to(cuda)
    v = ops.edge_vectors(p, l, sh.to(cuda), plan, ei[1].to(cuda), eg, ptr.to(cuda))
    got = torch.autograd.grad(v, [p, l], go.to(cuda))
    pr, lr = pos.double().requires_grad_(True), lat.double().requires_grad_(True)
    w = pr[ei[1]] - pr[ei[0]] + torch.einsum("ei,eij->ej", sh.double(), lr[batch[ei[0]]])
    want = torch.autograd.grad(w, [pr, lr], go.double())
    for a, b in zip(got, want):
        assert _rel(a.cpu(), b) < 20 * EPS[dtype]
    with pytest.raises(ValueError, match="numbers of graphs"):
        ops.edge_vectors(p, l, sh.to(cuda), plan, ei[1].to(cuda), eg, ptr[:3].to(cuda))


@pytest.mark.parametrize("n,n_keys,skew", [(0, 3, 0), (1, 1, 0), (300, 7, 0), (8192, 4096, 0), (8193, 4096, 0),
                                           (8192, 4097, 0), (30000, 50, 0), (30000, 9000, 1), (12345, 2, 0),
                                           (50000, 5, 1), (8192, 10, 1)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_group_keys_equals_stable_sort(cuda, n, n_keys, skew, dtype):
    """Both forms of the grouping (one workgroup, several launches), ranges
    longer than the ranked ones, strided keys, keys read through positions."""
    g = torch.Generator().manual_seed(n + n_keys)
    keys = torch.randint(0, n_keys, (n,), generator=g)
    if skew:   # most positions in one range
        keys[torch.rand(n, generator=g) < 0.8] = n_keys // 2
    wide = torch.stack([keys, torch.zeros_like(keys)], 1).to(dtype).to(cuda)
    perm = torch.randperm(n, generator=g)
    for k, through, ref in ((wide[:, 0], None, keys), (wide[:, 0].contiguous(), perm.to(torch.int32).to(cuda), keys[perm])):
        flags = torch.empty(2, dtype=torch.int32, device=cuda)
        k32, rp, order, _ = ops._group_keys(k, n_keys, through=through, flags=flags)
        assert torch.equal(k32.cpu(), ref.to(torch.int32))
        assert torch.equal(order.cpu().long(), torch.argsort(ref, stable=True))
        assert torch.equal(rp.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.int64),
                                                       torch.bincount(ref, minlength=n_keys).cumsum(0)]))
        assert flags.tolist() == [0, int(bool((ref[1:] < ref[:-1]).any()))]


@pytest.mark.parametrize("n", [50, 20000])
def test_edge_plan_refuses_nodes_out_of_range(cuda, n):
    """Negative and too large ids in either row are refused (the kernels skip
    them; nothing is indexed with them); int32 and column-major edge lists are
    taken."""
    g = torch.Generator().manual_seed(n)
    ei = torch.randint(0, 40, (2, n), generator=g)
    for row, bad in ((0, -1), (0, 40), (1, -3), (1, 2 ** 40)):
        e = ei.clone()
        e[row, n // 2] = bad
        with pytest.raises(ValueError, match="outside"):
            ops.EdgePlan.from_edge_index(e.to(cuda), 40)
    want = ops.EdgePlan.from_edge_index(ei, 40)   # the torch form, on the CPU
    for e in (ei.to(cuda), ei.to(torch.int32).to(cuda), ei.t().contiguous().to(cuda).t()):
        plan = ops.EdgePlan.from_edge_index(e, 40)
        for a, b in ((plan.rowptr, want.rowptr), (plan.src, want.src), (plan.eid, want.eid)):
            assert torch.equal(a.cpu(), b)
        for a, b in zip(plan.sender_csr(), want.sender_csr()):
            assert torch.equal(a.cpu(), b)


@pytest.mark.parametrize("m,k,n,bias", [(1, 32, 16, True), (63, 96, 384, True), (64, 33, 70, False), (129, 384, 96, True),
                                        (300, 768, 1152, True), (5001, 250, 129, False), (0, 64, 64, False)])
def test_gemm_bx3_and_layout_match_float64(cuda, m, k, n, bias):
    """Operands laid out from stacked, scaled weights (W^T and W, float32 and
    bf16, row-major floats) and the float32 product against float64: edges of
    the 64-row halves, the 128-column tiles, 32-k steps and 16-byte rows."""
    g = torch.Generator().manual_seed(m + k)
    cut = [n // 3, n - n // 3]
    W = [torch.randn(c, k, generator=g).to(cuda) for c in cut]
    alpha = [0.3, 1.7]
    seg = [v for w, c, a in zip(W, cut, alpha) for v in (w.data_ptr(), c, torch.tensor([a]).double().view(torch.int64).item())]
    pad = lambda r: r + [0] * (20 - len(r))
    nb = lambda a, b: 1024 * ((a + 31) // 32) * ((b + 15) // 16)
    sizes = [3 * nb(k, n), 3 * nb(n, k), nb(k, n), nb(n, k), 4 * n * k]
    offs = [sum((s + 15) // 16 * 16 for s in sizes[:i]) for i in range(6)]
    rows = [pad([1, k, n, offs[0], 2, 0, 1, k] + seg), pad([1, n, k, offs[1], 2, 1, 0, k] + seg),
            pad([0, k, n, offs[2], 2, 0, 1, k] + seg), pad([0, n, k, offs[3], 2, 1, 0, k] + seg),
            pad([2, n, k, offs[4], 2, 1, 0, k] + seg)]
    buf = ops.layout_operands(torch.tensor(rows, dtype=torch.int64, device=cuda), offs[5])
    full = torch.cat([w * torch.tensor(a, dtype=torch.float32) for w, a in zip(W, alpha)])   # [n, k]
    view = lambda i, dt: buf[offs[i]:offs[i] + sizes[i]].view(dt)
    assert torch.equal(view(4, torch.float32).view(n, k), full)
    assert torch.equal(view(2, torch.bfloat16), ops.bf16_fragment_order(full.t().to(torch.bfloat16)))
    assert torch.equal(view(3, torch.bfloat16), ops.bf16_fragment_order(full.to(torch.bfloat16)))
    x, go = torch.randn(m, k, generator=g).to(cuda), torch.randn(m, n, generator=g).to(cuda)
    b = torch.randn(n, generator=g).to(cuda) if bias else None
    y = ops.gemm_bx3(x, view(0, torch.int16), n, k, b)
    gx = ops.gemm_bx3(go, view(1, torch.int16), k, n)
    assert y.shape == (m, n) and gx.shape == (m, k)
    if m == 0:
        return
    want = x.double() @ full.double().t() + (b.double() if bias else 0.0)
    # 2^-24 of the running sum at each of its 6 k / 32 accumulations, and 2^-23 of each product left out
    tol = lambda kk: 2.0 ** -24 * (6 * kk / 32) ** 0.5 + 2.0 ** -23
    assert ((y.double() - want).norm() / want.norm()).item() < tol(k)
    want = go.double() @ full.double()
    assert ((gx.double() - want).norm() / want.norm()).item() < tol(n)


@pytest.mark.parametrize("n,most", [(1, 0), (1, 200), (5, 63), (7, 64), (300, 129)])
def test_edge_index_of_csr(cuda, n, most):
    """Senders and receivers of a receiver CSR: empty receivers, runs below,
    at and above a wavefront, a last group of receivers that is not full."""
    g = torch.Generator().manual_seed(n + most)
    counts = torch.randint(0, most + 1, (n,), generator=g)
    counts[n // 2] = most
    rowptr = torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)]).to(torch.int32)
    src = torch.randint(0, n, (int(counts.sum()),), generator=g, dtype=torch.int32)
    ei, dst = ops.edge_index_of(rowptr.to(cuda), src.to(cuda))
    want = torch.repeat_interleave(torch.arange(n), counts)
    assert ei.dtype == torch.int64 and dst.dtype == torch.int32
    assert torch.equal(ei.cpu(), torch.stack([src.to(torch.int64), want])) and torch.equal(dst.cpu().to(torch.int64), want)


@pytest.mark.parametrize("E,n", [(1, 5), (31, 260), (33, 768), (129, 2944), (1000, 36), (4097, 2944), (33000, 1000),
                                 (140000, 256)])
def test_last_radial_layer_parts(cuda, E, n):
    """Last layer and its input gradient (of edges and of pair rows, some
    alone): chunks and column parts of every length, remainders of 32 edges,
    128 rows and 32 columns.  At most six products per 16 terms are added one
    after another, each sum rounded once, and a part more."""
    g = torch.Generator().manual_seed(E + n)
    h, W, go = torch.randn(E, 64, generator=g), torch.randn(64, n, generator=g), torch.randn(E, n, generator=g)
    hc, Wc, gc = h.to(cuda), W.to(cuda), go.to(cuda)
    w64, u = W.double(), 2.0 ** -24
    rows = torch.cat([torch.arange(0, E, max(1, E // 400)), torch.tensor([E - 1])])
    got = ops.launch_mlp_out_f32(hc, Wc, 0.5).cpu()[rows].double()
    bound = (6 * 64 / 16 + 8) * u * 0.5 * (h[rows].double().abs() @ w64.abs())
    assert ((got - 0.5 * h[rows].double() @ w64).abs() <= bound).all()
    q, parts = ops._mlp_out_bwd_parts(E, n, cuda)
    assert (q == 1) == (parts is None) and (q - 1) * 32 * -(-((n + 31) // 32) // q) < n
    tol = (6 * n / 16 + 8 + q) * u * 0.5
    if n % 4 == 0:
        got = ops.launch_mlp_out_bwd_f32(gc, Wc, 0.5).cpu()[rows].double()
        assert ((got - 0.5 * go[rows].double() @ w64.t()).abs() <= tol * (go[rows].double().abs() @ w64.abs().t())).all()
    ra = torch.randperm(E, generator=g).to(torch.int32)
    rb = torch.where(torch.arange(E) % 7 == 0, -1, torch.randperm(E, generator=g)).to(torch.int32)
    pairs = ops.EdgePairs(E, ra.to(cuda), ra.to(cuda), rb.to(cuda))
    got = ops.launch_mlp_out_bwd_pairs_f32(gc, pairs, Wc, 0.5).cpu()[rows].double()
    a, b = go[ra[rows].long()], go[rb[rows].clamp_min(0).long()] * (rb[rows] >= 0)[:, None]
    s = a.double() + b.double()
    mag = (a.double().abs() + b.double().abs()) @ w64.abs().t()
    assert ((got - 0.5 * s @ w64.t()).abs() <= (tol + u) * mag).all()


@pytest.mark.parametrize("E,n_in,n,off", [(1, 8, 3, 0), (33, 7, 3, 0), (300, 32, 4, 0), (129, 1, 1, 0), (64, 10, 2, 1),
                                          (0, 8, 3, 0)])
def test_hidden_layers_scale_their_weights(cuda, E, n_in, n, off):
    """Weights scaled in the kernel and before it: the same bits, forward and
    input gradient (odd first layers, 1 .. 4 layers, matrices off 16 bytes)."""
    g = torch.Generator().manual_seed(E + n_in)
    mats = []
    for layer in range(n):
        buf = torch.empty((64 if layer else n_in) * 64 + off, device=cuda)
        mats.append(buf[off:].view(-1, 64).copy_(torch.randn(64 if layer else n_in, 64, generator=g)))
    scales = [(1.0 if layer == 0 else 2 ** 0.5) / m.shape[0] ** 0.5 for layer, m in enumerate(mats)]
    x = torch.randn(E, n_in, generator=g).to(cuda).requires_grad_(True)
    gh = torch.randn(E, 64, generator=g).to(cuda)
    a = ops.radial_mlp_hidden(x, mats, scales)
    b = ops.radial_mlp_hidden(x, [m * s for m, s in zip(mats, scales)])
    (ga,), (gb,) = torch.autograd.grad(a, x, gh), torch.autograd.grad(b, x, gh)
    assert torch.equal(a, b) and torch.equal(ga, gb)
    w = [m.double().cpu() * s for m, s in zip(mats, scales)]
    h = x.detach().double().cpu()
    for m in w:
        h = torch.nn.functional.silu(h @ m)
    assert E == 0 or (a.double().cpu() - h).abs().max() < 1e-5 * h.abs().max().clamp_min(1)


@pytest.mark.parametrize("n,box,rc", [(1, 3.0, 0.5), (1, 3.0, 6.0), (40, 6.0, 4.2), (260, 7.5, 4.0), (260, 7.5, 5.6)])
def test_neighbours_kept_or_searched_again(cuda, n, box, rc, monkeypatch):
    """Receivers with no neighbour, with fewer than the kept hits, around them
    and with more: copied, searched again and by a thread per receiver, the
    same edges in the same order."""
    g = torch.Generator().manual_seed(n)
    pos = (torch.rand(n, 3, generator=g, dtype=torch.float64) * box).to(cuda)
    cell = (box * torch.eye(3, dtype=torch.float64)).numpy()
    args = (pos, [n], [cell], [(True, True, False)], rc)
    kept, single = ops.neighbour_list_batch(*args), ops.neighbour_list(pos, cell, (True, True, False), rc)
    thread = ops.neighbour_list_batch(*args, mode=1)
    monkeypatch.setattr(ops, "NL_KEEP_ATOMS", 0)
    again = ops.neighbour_list_batch(*args)
    for other in (single, thread, again):
        assert all(torch.equal(a, b) for a, b in zip(kept, other))
    counts = kept[0].diff()
    if n == 260:
        over = counts > ops.NL_KEEP
        assert over.any() and bool((~over).any()) == (rc < 5)
