"""The forward's launch shapes: one output channel per workgroup with 4, 2 or 1 rows per wave (below 1024
workgroups of the full shape), the full shape, 9x9 elements, and the max / min winner rescans that go
with them (row by row from global memory, or by channel from LDS for up to 8 input channels).

Against the oracle: values bit for bit (zero signs included), winners exactly, gradients within the contract.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import TOL, normwise_error, seeded

pytestmark = pytest.mark.gpu

import morphocore_amd as mca  # noqa: E402
from morphocore_amd import _native  # noqa: E402

# (B, Cin, Cout, H, W): workgroups with 4 rows per wave around the shapes' limits (16-row tiles, one output
# channel): 448 and more, 192 of two rows and more, fewer.
SHAPES = [
    (2, 3, 7, 130, 200),  # 504 workgroups of four rows; bucket rescan
    (2, 9, 7, 130, 200),  # the same with more input channels than one channel's bucket takes
    (1, 10, 5, 70, 260),  # 225 of two rows
    (1, 2, 3, 17, 65),    # one row
    (3, 9, 4, 1, 70),     # a plane of one row
    (4, 2, 24, 129, 190),  # the full shape
]


@pytest.mark.parametrize("K", [3, 5, 7, 9, 11])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("op,merge,padding", [(0, "max", "replicate"), (1, "min", "geodesic"), (0, "min", "constant"), (1, "sum", "zero"), (0, "mean", "replicate")])
def test_forward_shapes(K, shape, op, merge, padding):
    B, Cin, Cout, H, W = shape
    if K * K * B * Cin * Cout * H * W > 2.5e8:
        pytest.skip("the oracle takes too long")
    pad, pv = {"zero": 0, "geodesic": 1, "constant": 2, "replicate": 3}[padding], -0.5
    # Quantised inputs: ties between taps and channels, zero results of either sign.
    x = seeded(31, B, Cin, H, W, kind="quant") - 0.5
    w = (seeded(32, Cout, Cin, K, K, kind="quant") * 4).round() / 4 - 0.5
    g = seeded(33, B, Cout, H, W, kind="randn")
    m = O.MERGES[merge]
    packed = merge in ("max", "min")
    ref, idx = O.morpho_forward(op, m, pad, pv, x.numpy(), w.numpy(), save_indices=packed)
    xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
    run = torch.ops.morphocore.dilation if op == 0 else torch.ops.morphocore.erosion
    out = run(xd, wd, m, pad, pv, True, 0.0)
    got = out.detach().cpu().numpy()
    assert np.array_equal(got, ref) and np.array_equal(np.signbit(got), np.signbit(ref))
    with torch.no_grad():
        assert np.array_equal(run(xd, wd, m, pad, pv, True, 0.0).cpu().numpy(), ref)  # values only
    if packed:
        o2, i2 = torch.empty_like(out), torch.empty(out.shape, dtype=torch.int32, device="cuda")
        fill = {"zero": 0.0, "geodesic": float("-inf") if op == 0 else float("inf"), "constant": pv, "replicate": 0.0}[padding]
        _native.morpho_forward(op, m, padding == "replicate", fill, xd.detach(), wd.detach(), 0, o2, i2, (B, Cin, Cout, Cin, H, W, K, K))
        assert np.array_equal(i2.cpu().numpy(), idx)
    out.backward(g.cuda())
    gx, gw = O.morpho_backward(op, m, pad, pv, x.numpy(), w.numpy(), g.numpy(), indices=idx if packed else None)
    assert normwise_error(xd.grad.cpu().numpy(), gx) <= TOL[torch.float32]
    assert normwise_error(wd.grad.cpu().numpy(), gw) <= TOL[torch.float32]


@pytest.mark.parametrize("K,merge,Cin", [(3, "max", 3), (5, "min", 4), (5, "max", 5), (7, "max", 8), (9, "min", 9), (11, "max", 4), (3, "sum", 3), (5, "mean", 2),
                                         (7, "sum", 2), (9, "mean", 2), (11, "sum", 2), (3, "identity", 0), (7, "identity", 0)])
@pytest.mark.parametrize("B,Cout,H,W", [
    (7, 14, 33, 60),   # 294 workgroups of four rows, 490 of two
    (13, 14, 30, 60),  # 364 and 728
    (12, 30, 40, 30),  # 1080 and 1800
    (90, 9, 8, 20),    # 810 of two rows; four would leave waves without rows
    (90, 9, 4, 20),    # planes of four rows: one row per wave
    (16, 3, 60, 200),  # three output channels: one per workgroup in the full shape too
])
def test_saving_forward_shapes(K, merge, Cin, B, Cout, H, W):
    """Rows per wave of the launches that save winners or taps, and the input channels up to which one output
    channel's winners are sorted (two a row per wave, one of 5x5): values and gradients."""
    Cin = Cin or Cout
    Cw = 1 if merge == "identity" else Cin
    x = seeded(51, B, Cin, H, W, kind="quant") - 0.5
    w = (seeded(52, Cout, Cw, K, K, kind="quant") * 4).round() / 4 - 0.5
    g = seeded(53, B, Cout, H, W, kind="randn")
    m = O.MERGES[merge]
    packed = merge in ("max", "min")
    ref, idx = O.morpho_forward(0, m, O.REPLICATE, 0.0, x.numpy(), w.numpy(), save_indices=packed)
    xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
    out = torch.ops.morphocore.dilation(xd, wd, m, O.REPLICATE, 0.0, True, 0.0)
    got = out.detach().cpu().numpy()
    assert np.array_equal(got, ref) and np.array_equal(np.signbit(got), np.signbit(ref))
    out.backward(g.cuda())
    gx, gw = O.morpho_backward(0, m, O.REPLICATE, 0.0, x.numpy(), w.numpy(), g.numpy(), indices=idx if packed else None)
    assert normwise_error(xd.grad.cpu().numpy(), gx) <= TOL[torch.float32]
    assert normwise_error(wd.grad.cpu().numpy(), gw) <= TOL[torch.float32]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("padding", ["geodesic", "replicate"])
def test_sixteen_bit_staging(dtype, padding):
    """16-bit tiles keep their storage type until they are staged; the fill value is float32."""
    x, w = seeded(41, 2, 5, 57, 57, dtype=dtype), seeded(42, 6, 5, 9, 9, dtype=dtype, kind="randn", scale=0.2)
    pad = {"geodesic": 1, "replicate": 3}[padding]
    ref = O.morpho_forward(0, O.MERGES["max"], pad, 0.0, x.float().numpy(), w.float().numpy())[0]
    out = torch.ops.morphocore.dilation(x.cuda(), w.cuda(), O.MERGES["max"], pad, 0.0, True, 0.0)
    assert np.array_equal(out.float().cpu().numpy(), torch.from_numpy(ref).to(dtype).float().numpy())
