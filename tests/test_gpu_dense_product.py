"""``tace_gemm_bx3`` on values at the ends of float32: the infinities and NaN of a float32 product (GPU)."""

import struct

import pytest
import torch

from tace_amd import ops

pytestmark = pytest.mark.gpu

MAX = torch.finfo(torch.float32).max
INF, NAN = float("inf"), float("nan")


def _product(x, W, bias, cuda):
    """x @ W on the kernel, W [k, n] laid out by ``tace_layout_operands``."""
    k, n = W.shape
    Wd = W.to(cuda).contiguous()
    size = 3 * 1024 * ((k + 31) // 32) * ((n + 15) // 16)
    row = [1, k, n, 0, 1, 0, 0, n, Wd.data_ptr(), n, struct.unpack("q", struct.pack("d", 1.0))[0]] + [0] * 9
    buf = ops.layout_operands(torch.tensor([row], dtype=torch.int64), size, cuda)
    return ops.gemm_bx3(x.to(cuda).contiguous(), buf.view(torch.int16), n, k, None if bias is None else bias.to(cuda)).cpu()


# where: (row of x, k, value) or (k, column of W, value)
SPECIAL = [("x", 5, 3, INF), ("x", 70, 95, -INF), ("x", 0, 0, NAN), ("w", 40, 17, INF), ("w", 99, 129, -INF),
           ("w", 1, 0, NAN), ("x", 5, 3, MAX), ("x", 130, 50, 3.39e38), ("w", 40, 17, -MAX), ("w", 40, 17, 3.396e38)]


@pytest.mark.parametrize("m,k,n", [(131, 100, 130), (65, 101, 131), (131, 96, 128)])
@pytest.mark.parametrize("bias", [False, True])
def test_infinities_of_a_float32_product(cuda, m, k, n, bias):
    """Each value alone, and all: finite where float64 stays in float32's
    range, else the same infinity or NaN; every other output as without them."""
    g = torch.Generator().manual_seed(m)
    x0, W0 = torch.randn(m, k, generator=g), torch.randn(k, n, generator=g) * 1e-3
    b = torch.randn(n, generator=g) if bias else None
    clean = _product(x0, W0, b, cuda)
    for special in [[s] for s in SPECIAL] + [SPECIAL]:
        x, W = x0.clone(), W0.clone()
        for where, i, j, v in special:
            t = x if where == "x" else W
            if i < t.shape[0] and j < t.shape[1]:
                t[i, j] = v
        got = _product(x, W, b, cuda)
        want64 = x.double() @ W.double() + (0 if b is None else b.double())
        want = want64.float()
        assert torch.equal(torch.isnan(got), torch.isnan(want)), special
        assert torch.equal(torch.isposinf(got), torch.isposinf(want)) and torch.equal(got == -INF, want == -INF), special
        fin = torch.isfinite(want)
        # k products rounded once each, and their sums, in one order or another
        size = x.double().abs().nan_to_num(0, 0, 0) @ W.double().abs().nan_to_num(0, 0, 0) + 1
        assert ((got.double() - want64).abs()[fin] <= (k + 2) * 2.0 ** -24 * size[fin]).all(), special
        rows = (x == x0).all(1)[:, None] & (W == W0).all(0)
        assert torch.equal(got[rows], clean[rows]), special


def test_all_inputs_not_finite(cuda):
    """Every output at once, also of the rows and columns past a tile: ends, and without a bias of its own."""
    for v, w in ((NAN, 1.0), (INF, 1.0), (INF, -1.0), (INF, 0.0), (1.0, INF)):
        x, W = torch.full((200, 384), v), torch.full((384, 150), w)
        got, want = _product(x, W, None, cuda), x @ W
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.nan_to_num(7), want.nan_to_num(7))
