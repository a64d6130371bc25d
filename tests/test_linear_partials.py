"""The partial tiles of segmented linears with k split over workgroups: bounded, whatever the size of the launch."""

import numpy as np
import pytest
import torch

from tace_amd import model as pm
from tace_amd import ops


@pytest.mark.parametrize("n", [3000, 20000])
def test_partial_tiles_are_bounded(n):
    """The coefficient linear of a correlation-3 product basis, 89 species, 256
    channels: its weights stream, so k is split at any number of nodes."""
    irr = pm.Irreps("5888x0e+8704x1o+10752x2e+10240x3o")
    lay = pm._LinearLayout(irr, pm.Irreps("256x0e+256x1o+256x2e+256x3o"))
    edges = np.sort(np.random.default_rng(n).integers(0, n, 88))
    rr = [(s, int(a), int(b)) for s, (a, b) in enumerate(zip([0, *edges], [*edges, n])) if b > a]
    weight = torch.empty(89, lay.weight_numel, device="meta")
    x = torch.empty(n, 1, device="meta")
    plan = lay.seg_plan("fwd", rr, n, x.new_empty(0, device="cpu"), weight, None)
    assert plan.splits > 1
    held = max(m for _, m in plan.launches) * plan.splits * 65536
    assert held <= 1.3 * ops.SEG_PARTIAL_BYTES   # runs of equal cost are padded to one length
    tiles = plan.tiles.numpy()
    assert sum(m for _, m in plan.launches) == plan.n_tiles == len(tiles)
    # every row and column of every output block once
    rows = tiles[tiles[:, 1] > 0]
    covered = (rows[:, 1] * np.minimum(128, rows[:, 2] - rows[:, 3])).sum()
    assert covered == n * 256 * 16 and len(np.unique(rows[:, [0, 3]], axis=0)) == len(rows)


@pytest.mark.parametrize("name,value", [
    ("SEG_KS_MIN_N", None), ("SEG_KS_CHUNK", {128: 256, 256: 1024}), ("SEG_TILE_FRAG", False), ("SEG_SPLIT_SLOTS", None),
    ("SEG_SPLIT_MIN_STEPS", 2), ("SEG_SPLIT_MAX_WORK", 0), ("SEG_STREAM_BYTES", 1 << 10), ("SEG_STREAM_STEPS", 4),
    ("SEG_PARTIAL_BYTES", 1 << 16), ("SEG_BALANCE_MIN", 1)])
def test_a_changed_setting_makes_another_plan(name, value, monkeypatch):
    lay = pm._LinearLayout(pm.Irreps("600x0e+90x1o"), pm.Irreps("160x0e+300x1o"))
    w, x = torch.empty(2, lay.weight_numel, device="meta"), torch.empty(0)
    rr = [(0, 0, 70), (1, 70, 200)]
    make = lambda: lay.seg_plan("fwd", rr, 200, x, w, None)
    first = make()
    assert make() is first
    with monkeypatch.context() as m:
        m.setattr(ops, name, value)
        assert make() is not first
    assert make() is first
    # the settings the plan reads, and no others
    assert {n for n in vars(ops) if n.startswith("SEG_")} == {"SEG_KS_MIN_N", "SEG_KS_CHUNK", "SEG_TILE_FRAG", "SEG_SPLIT_SLOTS",
            "SEG_SPLIT_MIN_STEPS", "SEG_SPLIT_MAX_WORK", "SEG_STREAM_BYTES", "SEG_STREAM_STEPS", "SEG_PARTIAL_BYTES",
            "SEG_BALANCE_MIN"}


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", [1, 7, 64, 100])
def test_several_launches_give_the_bits_of_one(cuda, tiles, monkeypatch):
    """Launches of few tiles and of more than the equal-cost runs start at,
    with an addend apart and in place."""
    counts = [1, 33, 64, 65, 130, 257, 0] * 4
    S, Z = len(counts), sum(counts)
    species = torch.repeat_interleave(torch.arange(S), torch.tensor(counts))
    g = torch.Generator().manual_seed(3)
    lin = pm.e3nnElementLinear("1100x0e+900x1o", "160x0e+100x1o", S).to(cuda).requires_grad_(False)
    sp = pm.SpeciesPlan(torch.nn.functional.one_hot(species, S).float().to(cuda))
    x, add = torch.randn(Z, lin.lay.dim_in, generator=g).to(cuda), torch.randn(Z, lin.lay.dim_out, generator=g).to(cuda)
    rr, seg = pm._linear_route(x, lin.weight, lin.lay, sp.ranges)
    monkeypatch.setattr(ops, "SEG_STREAM_BYTES", 1 << 20)
    monkeypatch.setattr(ops, "SEG_STREAM_STEPS", 8)
    monkeypatch.setattr(ops, "SEG_SPLIT_MAX_WORK", 0)
    monkeypatch.setattr(ops, "SEG_SPLIT_MIN_STEPS", 1)
    res = []
    for limit in (1 << 40, tiles * 4 * 65536):
        monkeypatch.setattr(ops, "SEG_PARTIAL_BYTES", limit)
        y = pm._linear_apply(x, lin.weight, lin.bias, lin.lay, rr, seg, 0.9, out=None, addend=add)
        z = add.clone()
        pm._linear_apply(x, lin.weight, lin.bias, lin.lay, rr, seg, 0.9, out=z, addend=z)
        res.append((y, z))
        plan = lin.lay.seg_plan("fwd", rr, Z, x, lin.weight, lin.bias)
        assert plan.splits == 4 and (len(plan.launches) > 1) == (limit < 1 << 40)
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
