"""grad_input summed by tiles in LDS (morpho_scatter.hip), at the edges of its plans.

Max / min past the small problems' gather: one tile column and several, channel groups of more than 64
input channels, elements larger than the tile, partial last tiles, and an element so large for its channel
count that the global atomics stay. Identity in float32 and 16-bit on planes the row bands do not take:
one to two tile columns, planes of one row or column, even, rectangular and 17x17 elements (two-byte
taps). Against the oracle: the operator's contract (1e-6 / 1e-12, one rounding in 16 bits).

Backwards without saved taps walk the batch in chunks over one layout of partial slots: at shapes whose
tiles depend on the batch, and chunks that do not divide it.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import TOL, normwise_error, seeded

pytestmark = pytest.mark.gpu

import morphocore_amd as mca  # noqa: E402

GTOL = {**TOL, torch.float16: 1e-3, torch.bfloat16: 8e-3}


def _run(op, merge, padding, dtype, B, Cin, Cout, H, W, KH, KW):
    Cw = 1 if merge == "identity" else Cin
    x = seeded(11, B, Cin, H, W, dtype=dtype)
    w = seeded(12, Cout, Cw, KH, KW, dtype=dtype, kind="randn", scale=0.1)
    g = seeded(13, B, Cout, H, W, dtype=dtype, kind="randn")
    g[:, :, ::3, ::5] = 0.0
    xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
    run = torch.ops.morphocore.dilation if op == "dilation" else torch.ops.morphocore.erosion
    out = run(xd, wd, O.MERGES[merge], {"zero": 0, "geodesic": 1, "replicate": 3}[padding], 0.0, True, 0.0)
    out.backward(g.cuda())
    ref_t = torch.float64 if dtype == torch.float64 else torch.float32
    xr, wr, gr = (t.to(ref_t).numpy() for t in (x, w, g))
    o, pad = (O.DILATION if op == "dilation" else O.EROSION), {"zero": 0, "geodesic": 1, "replicate": 3}[padding]
    idx = O.morpho_forward(o, O.MERGES[merge], pad, 0.0, xr, wr, save_indices=True)[1] if merge in ("max", "min") else None
    gx, gw = O.morpho_backward(o, O.MERGES[merge], pad, 0.0, xr, wr, gr, indices=idx)
    for name, got, want in (("grad_input", xd.grad, gx), ("grad_weight", wd.grad, gw)):
        err = normwise_error(got.float().cpu().numpy() if dtype in (torch.float16, torch.bfloat16) else got.cpu().numpy(), want)
        assert err <= GTOL[dtype], f"{name}: {err}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", [
    (1, 3, 8, 200, 300, 5, 5),     # several 64-wide tiles, partial last ones
    (2, 65, 16, 33, 65, 3, 3),     # two channel groups
    (1, 64, 3, 57, 57, 11, 11),    # 64 channels: tiles smaller than the element's halo
    (3, 1, 40, 64, 300, 3, 7),     # one channel, rectangular element
    (1, 2, 4, 40, 300, 21, 21),    # tap numbers past 256
    (1, 2, 16, 1, 45000, 1, 31),   # a plane of one row
    (1, 130, 4, 31, 33, 9, 9),     # three channel groups
    (2500, 8, 16, 4, 5, 3, 3),     # small planes: winners walked across batch elements
])
def test_packed_tiles(shape, dtype):
    _run("erosion" if shape[1] % 2 else "dilation", "max" if shape[2] % 3 else "min", "replicate", dtype, *shape)


def test_packed_falls_back_to_atomics():
    _run("dilation", "max", "zero", torch.float32, 1, 128, 1, 80, 80, 41, 41)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("op,shape", [
    ("dilation", (2, 3, 3, 37, 29, 3, 3)),
    ("erosion", (1, 2, 2, 70, 257, 5, 5)),    # two tile columns
    ("dilation", (1, 1, 1, 130, 1030, 3, 3)),  # five
    ("erosion", (3, 5, 5, 1, 63, 7, 7)),      # one row
    ("dilation", (2, 4, 4, 300, 1, 5, 5)),    # one column
    ("erosion", (40, 30, 30, 13, 11, 4, 2)),  # one tile per plane, full-height tiles
    ("dilation", (1, 2, 2, 50, 47, 17, 17)),  # two-byte taps
    ("erosion", (1, 3, 3, 64, 100, 1, 9)),
    ("dilation", (3, 4, 4, 16, 16, 5, 5)),    # 256 pixels: one wave a tile
    ("erosion", (3, 4, 4, 16, 17, 5, 5)),     # four
    ("dilation", (50, 7, 7, 3, 2, 3, 3)),
])
def test_identity_tiles(op, shape, dtype):
    for padding in ("replicate", "geodesic"):
        _run(op, "identity", padding, dtype, *shape)


@pytest.mark.parametrize("op,shape,dtype", [
    ("dilation", (64, 32, 64, 64, 3, 3), torch.float32),   # 1 tile a plane for the batch, 16 for one element
    ("erosion", (16, 8, 128, 128, 5, 5), torch.float32),   # 4 and 32
    ("dilation", (16, 8, 128, 128, 7, 7), torch.float64),
])
def test_identity_recomputed_taps_in_chunks_of_one_plan(op, shape, dtype, monkeypatch):
    """Chunks of the batch take the tiles of the whole batch, which its partial slots are laid out by: the
    gradients are the oracle's, and the same bit for bit whatever the chunk (the gradient's values are
    multiples of 1/8 below 32, so that every sum of them is exact)."""
    B, C, H, W, KH, KW = shape
    x = seeded(14, B, C, H, W, dtype=dtype)
    w = seeded(15, C, 1, KH, KW, dtype=dtype, kind="randn", scale=0.1)
    g = (seeded(16, B, C, H, W, dtype=dtype, kind="randn") * 8).round() / 8
    o = O.DILATION if op == "dilation" else O.EROSION
    run = torch.ops.morphocore.dilation if op == "dilation" else torch.ops.morphocore.erosion
    one = C * H * W * (1 + x.element_size())  # taps and scratch output of one batch element
    gx, gw = O.morpho_backward(o, O.MERGES["identity"], O.REPLICATE, 0.0, x.numpy(), w.numpy(), g.numpy())
    grads = []
    for elements in (B, 1, 3, B - 1):
        monkeypatch.setenv("MORPHOCORE_AMD_RECOMPUTE_BYTES", str(elements * one))
        xd, wd = x.cuda().requires_grad_(), w.cuda().requires_grad_()
        run(xd, wd, O.MERGES["identity"], O.REPLICATE, 0.0, False, 0.0).backward(g.cuda())
        grads.append((xd.grad, wd.grad))
        assert normwise_error(xd.grad.cpu().numpy(), gx) <= TOL[dtype], elements
        assert normwise_error(wd.grad.cpu().numpy(), gw) <= TOL[dtype], elements
    for gi, wi in grads[1:]:
        assert torch.equal(gi, grads[0][0]) and torch.equal(wi, grads[0][1])
