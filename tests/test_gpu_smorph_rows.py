"""The smorph forward of launches with few workgroups (four waves, four input channels), whose values are the
reference's bit for bit, and the backward behind it: channel counts that are no multiple of four, planes
narrower than a wave, rows of several widths, launches on both sides of the limit. (The output-channel
slices of the generic backward: test_gpu_smorph_generic.py.)
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import TOL, normwise_error, seeded

pytestmark = pytest.mark.gpu

import morphocore_amd as mca  # noqa: E402,F401

SHAPES = [
    (torch.float32, (1, 5, 3, 9, 17, 3, 3)),      # three rows of 17 columns per wave
    (torch.float32, (2, 2, 2, 7, 16, 5, 5)),      # four rows of 16
    (torch.float32, (1, 3, 2, 1, 1, 5, 5)),       # one pixel
    (torch.float32, (1, 6, 2, 13, 65, 7, 7)),     # two strips of 33 columns
    (torch.float32, (1, 4, 1, 12, 64, 11, 11)),   # one row of 64, a tile inside the image
    (torch.float32, (1, 9, 2, 23, 130, 9, 9)),    # no saved statistics
    (torch.float64, (2, 3, 2, 11, 33, 3, 3)),
    (torch.float64, (1, 8, 3, 10, 60, 5, 5)),
    (torch.float64, (1, 5, 2, 25, 128, 11, 11)),
    (torch.float32, (1, 4, 10, 128, 64, 3, 3)),   # 1280 waves: this kernel
    (torch.float32, (1, 4, 10, 129, 64, 3, 3)),   # 1290: the other
    (torch.float32, (2, 4, 100, 14, 28, 3, 3)),   # above 1280, half the waves of the other: this kernel
    (torch.float32, (2, 5, 100, 14, 28, 3, 3)),   # with waves idle in the channels: the other
    (torch.float64, (2, 5, 8, 65, 64, 3, 3)),     # 1664 waves: this kernel
    (torch.float64, (1, 4, 48, 128, 64, 3, 3)),   # 6144: this kernel
    (torch.float64, (1, 4, 48, 129, 64, 3, 3)),   # 6192: the other
    (torch.float32, (1, 2, 8, 12, 40, 11, 11)),   # two input channels: the static kernels
    (torch.float32, (1, 2, 9, 12, 40, 7, 7)),
    (torch.float32, (1, 2, 11, 12, 40, 5, 5)),
    (torch.float32, (1, 2, 29, 12, 40, 3, 3)),
]


@pytest.mark.parametrize("saved", [True, False], ids=["saved-stats", "recomputed"])
@pytest.mark.parametrize("merge", ["sum", "mean", "max", "min"])
@pytest.mark.parametrize("dtype,shape", SHAPES, ids=[str(s[0])[6:] + "-" + "x".join(map(str, s[1])) for s in SHAPES])
def test_rows_forward_and_backward(dtype, shape, merge, saved, monkeypatch):
    if not saved and (dtype == torch.float64 or shape[-1] == 9):
        pytest.skip("no statistics are saved for this element")
    monkeypatch.setenv("MORPHOCORE_AMD_SAVED_STATS_LIMIT", "-1" if saved else "0")
    B, Cin, Cout, H, W, KH, KW = shape
    x = seeded(71, B, Cin, H, W, dtype=dtype, kind="randn")
    w = seeded(72, Cout, Cin, KH, KW, dtype=dtype, kind="randn", scale=0.2)
    alpha = seeded(73, Cout, Cin, dtype=dtype, kind="randn", scale=2.0)
    alpha[0, 0] = 0.0
    g = seeded(74, B, Cout, H, W, dtype=dtype, kind="randn")
    m = O.MERGES[merge]
    with torch.no_grad():
        plain = torch.ops.morphocore.smorph(x.cuda(), w.cuda(), alpha.cuda(), m)
    xd, wd, ad = (t.cuda().requires_grad_() for t in (x, w, alpha))
    out = torch.ops.morphocore.smorph(xd, wd, ad, m)
    out.backward(g.cuda())
    ref = O.smorph_forward(m, x.numpy(), w.numpy(), alpha.numpy())
    assert np.array_equal(plain.cpu().numpy(), ref)
    assert np.array_equal(out.detach().cpu().numpy(), ref)
    gx, gw, ga = O.smorph_backward(m, x.numpy(), w.numpy(), alpha.numpy(), g.numpy())
    for got, want in ((xd.grad, gx), (wd.grad, gw), (ad.grad, ga)):
        assert normwise_error(got.cpu().numpy().reshape(np.shape(want)), want) <= TOL[dtype]
