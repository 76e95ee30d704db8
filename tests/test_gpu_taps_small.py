"""Sum / mean backwards of few workgroups (8-row tiles, elements of 9 rows and more): every grad_input pixel is the
sum of several tiles, kept in double and rounded once.
"""
import pytest
import torch

from oracle import oracle as O
from tests.helpers import seeded

pytestmark = pytest.mark.gpu

import morphocore_amd as mca  # noqa: E402,F401


@pytest.mark.parametrize("merge", ["sum", "mean"])
@pytest.mark.parametrize("K", [9, 11, 17])  # (17: two-byte taps)
def test_tiles_that_cancel_leave_the_rest_exact(K, merge):
    """Outputs of two tiles with opposite gradients of 2^20 k reach the same input pixels (peaks that every
    window around them selects); what is left are sums of multiples of 1/16, exact in double. A float32
    sum per tile would round them to multiples of 1/8 and more."""
    B, Cin, Cout, H, W, peak = 1, 2, 3, 24, 4 * K, 10
    x = seeded(91, B, Cin, H, W)
    x[:, :, peak, K // 2::K] = 100.0
    w = seeded(92, Cout, Cin, K, K, kind="randn", scale=0.1)
    small = seeded(93, B, Cout, H, W, kind="quant")
    small[:, :, peak - 4:peak] = 0.0
    large = torch.zeros_like(small)
    large[:, :, peak - 4:peak - 2] = 2.0 ** 24 * seeded(94, B, Cout, 2, W, kind="quant")  # rows 6 and 7: tile 0
    large[:, :, peak - 2:peak] = -large[:, :, peak - 4:peak - 2]                           # rows 8 and 9: tile 1
    grads = []
    for g in (small, small + large):
        xd = x.cuda().requires_grad_()
        torch.ops.morphocore.dilation(xd, w.cuda(), O.MERGES[merge], O.REPLICATE, 0.0, True, 0.0).backward(g.cuda())
        grads.append(xd.grad)
    assert torch.equal(*grads)
