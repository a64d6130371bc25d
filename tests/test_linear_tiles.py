"""Segmented linears: tiles run as two 64-row halves, tables in XCD runs of equal cost."""

import numpy as np
import pytest
import torch

from tace_amd import ops


@pytest.mark.parametrize("n,spread,nruns", [(64, 1, 8), (100, 40, 4), (1537, 9, 8), (8, 3, 8), (2000, 400, 2), (70, 5, 1)])
def test_xcd_runs_keep_every_entry_and_share_the_cost(n, spread, nruns):
    """Every entry once, the rest zero rows; no run above the mean by more than its costliest entry."""
    rng = np.random.default_rng(n)
    table = np.stack([np.arange(n), rng.integers(1, 129, n), rng.integers(0, 9, n)], 1)
    cost = rng.integers(1, spread + 1, n)
    length = rng.integers(1, 4, n)
    out = ops._xcd_balanced(table, cost, length, nruns)
    assert len(out) % nruns == 0
    kept = out[out[:, 1] > 0]
    assert np.array_equal(kept[np.argsort(kept[:, 0])], table)
    assert (out[out[:, 1] == 0] == 0).all()
    runs = [r[r[:, 1] > 0][:, 0] for r in out.reshape(nruns, -1, 3)]
    assert max(cost[r].sum() for r in runs) <= cost.sum() / nruns + cost.max()
    for r in runs:
        assert (np.diff(length[r]) <= 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("irr_in,irr_out", [("96x0e+64x1o", "160x0e+32x1o"),       # short and odd k, two column tiles
                                            ("1100x0e+36x1o", "40x0e+300x1o"),     # long k; a short-k wide block
                                            ("30x0e+30x1o", "50x0e+300x1o")])      # rows of x off 16-byte boundaries
def test_seg_linear_row_halves_equal_in_kernel_split(cuda, irr_in, irr_out, monkeypatch):
    """Species of 1 .. 257 rows (ends of a 32-row block, of a half and of a
    tile), enough of them for tables in equal-cost runs: the same bits as the
    kernel that keeps whole tiles and splits the weights itself, forward and
    input gradient, with an addend in place."""
    from tace_amd import model as pm
    monkeypatch.setattr(pm, "SEG_LINEAR_TILE_F32", 128)
    monkeypatch.setattr(ops, "SEG_SPLIT_SLOTS", None)   # split k sums in another order
    monkeypatch.setattr(ops, "SEG_KS_MIN_N", 256)       # the tile kernel for narrow blocks
    counts = [1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 191, 192, 193, 257, 0] * 3
    S, Z = len(counts), sum(counts)
    species = torch.repeat_interleave(torch.arange(S), torch.tensor(counts))
    g = torch.Generator().manual_seed(7)
    lin = pm.e3nnElementLinear(irr_in, irr_out, S)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(lin.weight.shape, generator=g))
        lin.bias.copy_(torch.randn(lin.bias.shape, generator=g))
    lin = lin.to(cuda).requires_grad_(False)
    sp = pm.SpeciesPlan(torch.nn.functional.one_hot(species, S).float().to(cuda))
    for kind, din, dout in (("fwd", lin.lay.dim_in, lin.lay.dim_out), ("bwd", lin.lay.dim_out, lin.lay.dim_in)):
        x, add = torch.randn(Z, din, generator=g).to(cuda), torch.randn(Z, dout, generator=g).to(cuda)
        rr, seg = pm._linear_route(x, lin.weight, lin.lay, sp.ranges)
        res = []
        for presplit in (False, True):
            monkeypatch.setattr(pm, "SEG_LINEAR_PRESPLIT", presplit)
            y = pm._linear_apply(x, lin.weight, lin.bias, lin.lay, rr, seg, 1.0, kind=kind)
            z = add.clone()
            pm._linear_apply(x, lin.weight, lin.bias, lin.lay, rr, seg, 1.0, kind=kind, out=z, addend=z)
            res.append((y, z))
        plan = lin.lay.seg_plan(kind, rr, Z, x, lin.weight, lin.bias if kind == "fwd" else None)
        assert plan.tile_frag and plan.n_tiles % 8 == 0 and plan.n_tiles >= ops.SEG_BALANCE_MIN
        assert torch.equal(res[1][0], res[0][0]), kind
        # the fragment-order kernels start their sums from the addend
        assert ((res[1][1] - res[0][1]).abs().max() / res[0][1].abs().max()).item() < 2e-6, kind


@pytest.mark.gpu
@pytest.mark.parametrize("steps,want", [(2, 8), (8, 4), (17, 2)])
def test_seg_linear_streamed_weights_split(cuda, steps, want, monkeypatch):
    """Weights beyond the cache limit (lowered here) with k split over runs of
    the whole table: equal to the unsplit launch up to float32 summation
    order, the same bits on a repeat."""
    from tace_amd import model as pm
    counts = [1, 33, 64, 65, 130, 257, 0] * 4
    S, Z = len(counts), sum(counts)
    species = torch.repeat_interleave(torch.arange(S), torch.tensor(counts))
    g = torch.Generator().manual_seed(3)
    lin = pm.e3nnElementLinear("1100x0e+900x1o", "160x0e+100x1o", S).to(cuda).requires_grad_(False)
    sp = pm.SpeciesPlan(torch.nn.functional.one_hot(species, S).float().to(cuda))
    x, add = torch.randn(Z, lin.lay.dim_in, generator=g).to(cuda), torch.randn(Z, lin.lay.dim_out, generator=g).to(cuda)
    rr, seg = pm._linear_route(x, lin.weight, lin.lay, sp.ranges)
    run = lambda: pm._linear_apply(x, lin.weight, lin.bias, lin.lay, rr, seg, 0.9, out=None, addend=add)
    monkeypatch.setattr(ops, "SEG_SPLIT_MAX_WORK", 0)
    ref = run()
    monkeypatch.setattr(ops, "SEG_STREAM_BYTES", 1 << 20)
    monkeypatch.setattr(ops, "SEG_STREAM_STEPS", steps)
    monkeypatch.setattr(ops, "SEG_SPLIT_MIN_STEPS", 1)
    got = run()
    plan = lin.lay.seg_plan("fwd", rr, Z, x, lin.weight, lin.bias)
    assert plan.splits == want and plan.n_tiles % (8 // want) == 0 and plan.n_tiles >= ops.SEG_BALANCE_MIN
    assert torch.equal(got, run())
    # k = 1100 products of unit variance in another order: 2^-24 sqrt(k) each way
    assert ((got - ref).abs().max() / ref.abs().max()).item() < 4e-6


@pytest.mark.parametrize("d,R", [(1, 64), (3, 64), (7, 128)])
def test_row_tiles_of_every_range(d, R):
    """Range by range, in order: no tile crosses a range, the last of each holds its remainder."""
    counts, rng, at = [1, 63, 64, 65, 0, 200], [], 0
    for s, c in enumerate(counts):
        rng.append((s if s else -1, at, at + c))
        at += c
    want = [(r, min(b * d - r, R), max(s, 0)) for s, a, b in rng for r in range(a * d, b * d, R)]
    got = ops.SegLinearPlan._row_tiles(np.array(rng, dtype=np.int64), d, R)
    assert [tuple(map(int, v)) for v in zip(*got)] == want
    assert all(len(v) == 0 for v in ops.SegLinearPlan._row_tiles(np.zeros((0, 3), np.int64), d, R))


def test_stacked_values_of_structures():
    """The quick form and the item by item one give the same array and refuse the same items."""
    cell = lambda c: c.reshape(3, 3)
    flag = lambda p: np.broadcast_to(p, (3,))
    c = np.arange(18, dtype=np.float64).reshape(2, 3, 3)
    for items in (list(c), list(c.reshape(2, 9)), c.tolist(), [c[0], c[1].ravel()], list(torch.from_numpy(c)), c):
        assert np.array_equal(ops._stacked(items, np.float64, (3, 3), cell), c)
    want = np.array([[1, 1, 0], [1, 1, 1]], dtype=np.int32)
    for items in ([(True, True, False), True], [[1, 1, 0], [1]], want.tolist(), list(torch.from_numpy(want))):
        got = ops._stacked(items, np.int32, (3,), flag)
        assert got.dtype == np.int32 and np.array_equal(got, want)
    for items, dtype, shape, one in (([], np.float64, (3, 3), cell), ([np.zeros((3, 2))], np.float64, (3, 3), cell),
                                     ([1.0], np.float64, (3, 3), cell), ([np.ones((3, 1))], np.int32, (3,), flag)):
        with pytest.raises(ValueError):
            ops._stacked(items, dtype, shape, one)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [5, 12, 32, 40, 96, 128, 130, 232, 256])
def test_short_k_tasks_equal_the_tile_kernel(cuda, k, monkeypatch):
    """Wide blocks of one contribution: tasks of 1 .. 64 rows (32 and fewer
    multiply half a tile), k around the 32-k steps and off the 8-k loads,
    column chunks with a remainder off the 32 columns: the bits of the kernel
    that keeps whole tiles, with a bias, and with an addend up to rounding.
    An infinity in one row stays in that row."""
    from tace_amd import model as pm
    counts = [1, 31, 32, 33, 0, 64, 65, 97, 150] * 4
    S, Z = len(counts), sum(counts)
    g = torch.Generator().manual_seed(k)
    lin = pm.e3nnElementLinear(f"{k}x0e+{k}x1o", "1093x0e+300x1o", S)
    with torch.no_grad():
        lin.weight.copy_(torch.randn(lin.weight.shape, generator=g))
        lin.bias.copy_(torch.randn(lin.bias.shape, generator=g))
    lin = lin.to(cuda).requires_grad_(False)
    species = torch.repeat_interleave(torch.arange(S), torch.tensor(counts))
    sp = pm.SpeciesPlan(torch.nn.functional.one_hot(species, S).float().to(cuda))
    x = torch.randn(Z, lin.lay.dim_in, generator=g).to(cuda)
    add = torch.randn(Z, lin.lay.dim_out, generator=g).to(cuda)
    x.view(-1)[3 * k + 1] = float("inf")   # node 3 of the first block
    rr, seg = pm._linear_route(x, lin.weight, lin.lay, sp.ranges)
    assert seg
    res = []
    for min_n in (None, 256):
        monkeypatch.setattr(ops, "SEG_KS_MIN_N", min_n)
        plan = lin.lay.seg_plan("fwd", rr, Z, x, lin.weight, lin.bias)
        assert (plan.n_ks > 0) == (min_n is not None)
        y = pm._linear_apply(x, lin.weight, lin.bias, lin.lay, rr, seg, 0.5)
        z = pm._linear_apply(x, lin.weight, lin.bias, lin.lay, rr, seg, 0.5, out=add.clone(), addend=add)
        res.append((y, z))
    (y0, z0), (y1, z1) = res
    bad = ~torch.isfinite(y0)
    assert int(bad.sum()) == 1093 and torch.equal(bad, ~torch.isfinite(y1)) and torch.equal(bad, ~torch.isfinite(z1))
    y0, y1, z0, z1 = (v[~bad] for v in (y0, y1, z0, z1))
    assert torch.equal(y0, y1)
    # sums started from the addend or ended with it: a rounding each of sums of k <= 256 products
    assert ((z1 - z0).abs().max() / z0.abs().max()).item() < 2e-6
