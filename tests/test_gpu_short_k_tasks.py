"""Tasks the short-k kernel is not built for come out as NaN, not as part of a product (GPU)."""

import pytest
import torch

from tace_amd import _native as N
from tace_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k_max,k,rows", [(128, 96, 128), (128, 128, 65), (256, 200, 100), (128, 160, 64), (256, 256, 64)])
def test_tall_and_deep_tasks(cuda, k_max, k, rows):
    """One task of the given height and depth, one of 64 rows behind it: the
    first NaN in all its rows (128 of them in the table of an older caller)
    where the kernel does not hold it, the second a product."""
    n, k2 = 150, min(k, k_max)
    g = torch.Generator().manual_seed(k)
    w1, w2 = torch.randn(k, n, generator=g).to(cuda), torch.randn(k2, n, generator=g).to(cuda)
    size = lambda kk: 3 * ((n + 15) // 16 * 16) * ((kk + 31) // 32 * 32)
    flat = torch.cat([w1.view(-1), w2.view(-1)])
    frag = ops.bf16x3_split_blocks(flat, [(0, n, k, 1, 0, 1), (k * n, n, k2, 1, size(k), 1)], [1.0, 1.0],
                                   size(k) + size(k2), frag=True)
    x = torch.randn(rows * k + 64 * k2, generator=g).to(cuda)
    y = torch.zeros((rows + 64) * n, device=cuda)
    tasks = torch.tensor([[0, rows, n, 0, n, -1, 0, k, 0, 0], [rows * n, 64, n, 0, n, -1, rows * k, k2, size(k), 0]],
                         dtype=torch.int64, device=cuda)
    N.check(N.lib().tace_seg_linear_presplit_ks(x.data_ptr(), y.data_ptr(), None, frag.data_ptr(), None,
                                                tasks.data_ptr(), 2, k_max, 1.0, N.stream_ptr(cuda)))
    first, second = y[:rows * n].view(rows, n), y[rows * n:].view(64, n)
    x1, x2 = x[:rows * k].view(rows, k).double(), x[rows * k:].view(64, k2).double()
    # six rounded sums per 32 products, none above the sum of the magnitudes, and
    # 2^-23 of each product left out
    close = lambda a, u, v: ((a.double() - u @ v.double()).abs()
                             <= (6 * len(v) / 32 + 2) * 2.0 ** -24 * (u.abs() @ v.double().abs())).all()
    assert close(second, x2, w2)
    if rows > 64 or k > k_max:
        assert torch.isnan(first).all()
    else:
        assert close(first, x1, w1)
