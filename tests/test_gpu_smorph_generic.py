"""The generic smorph kernels' unrolled rows (float64, and float32 elements without static kernels) and their
output-channel slices, on planes with tiles inside the image and at its edges; and the element blend
(torch.ops.morphocore.smorph_element) against the torch operations it replaces, bit for bit.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import TOL, normwise_error, seeded

pytestmark = pytest.mark.gpu

import morphocore_amd as mca  # noqa: E402
from morphocore_amd.functional.smorph import element, w_tilde  # noqa: E402


@pytest.mark.parametrize("merge", ["sum", "mean", "max", "identity"])
@pytest.mark.parametrize("dtype,shape", [
    (torch.float64, (1, 2, 5, 13, 200, 5, 5)),   # one slice per output channel
    (torch.float64, (2, 3, 7, 40, 150, 3, 3)),
    (torch.float64, (1, 1, 1, 9, 64, 7, 7)),
    (torch.float64, (1, 2, 3, 21, 140, 11, 11)),
    (torch.float32, (1, 3, 5, 33, 210, 9, 9)),
    (torch.float32, (2, 2, 3, 30, 130, 4, 5)),   # even height
    (torch.float32, (1, 2, 4, 1, 70, 3, 7)),     # a plane of one row
    (torch.float32, (40, 8, 6, 8, 70, 5, 3)),    # enough tiles: one slice
    # Output-channel slices of several channels (1024 workgroups over 16 planes of 8 strips: 8 slices):
    (torch.float64, (2, 8, 20, 32, 60, 5, 5)),   # six slices of three channels and one of two
    (torch.float64, (2, 8, 21, 32, 60, 3, 3)),   # seven of three
    (torch.float32, (2, 8, 20, 32, 60, 9, 9)),
    (torch.float32, (2, 8, 21, 32, 60, 5, 3)),
    (torch.float64, (1, 2, 3, 20, 70, 6, 6)),    # not unrolled
    (torch.float32, (1, 3, 2, 7, 21, 13, 13)),   # not unrolled, most taps outside the image
])
def test_generic_kernels(dtype, shape, merge):
    B, Cin, Cout, H, W, KH, KW = shape
    Cout = Cin if merge == "identity" else Cout
    Cw = 1 if merge == "identity" else Cin
    x = seeded(51, B, Cin, H, W, dtype=dtype, kind="randn")
    w = seeded(52, Cout, Cw, KH, KW, dtype=dtype, kind="randn", scale=0.2)
    alpha = seeded(53, Cout, Cw, dtype=dtype, kind="randn", scale=2.0)
    alpha[0, 0] = 0.0
    g = seeded(54, B, Cout, H, W, dtype=dtype, kind="randn")
    m = O.MERGES[merge]
    xd, wd, ad = (t.cuda().requires_grad_() for t in (x, w, alpha))
    out = torch.ops.morphocore.smorph(xd, wd, ad, m)
    out.backward(g.cuda())
    a_np = alpha.numpy() if merge != "identity" else alpha.numpy().reshape(-1)
    ref = O.smorph_forward(m, x.numpy(), w.numpy(), a_np)
    assert np.array_equal(out.detach().cpu().numpy(), ref)
    gx, gw, ga = O.smorph_backward(m, x.numpy(), w.numpy(), a_np, g.numpy())
    for got, want in ((xd.grad, gx), (wd.grad, gw), (ad.grad, ga)):
        assert normwise_error(got.cpu().numpy().reshape(np.shape(want)), want) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("mode,wshape,ashape", [("sum", (4, 3, 5, 5), (4, 3)), ("mean", (1, 1, 1, 1), (1, 1)), ("identity", (7, 1, 11, 11), (7, 1)),
                                                ("identity", (5, 1, 3, 4), (5,)), ("sum", (6, 1, 9, 9), (6,))])
def test_element_matches_torch(dtype, mode, wshape, ashape):
    w = seeded(61, *wshape, dtype=dtype, kind="randn").cuda()
    alpha = seeded(62, *ashape, dtype=dtype, kind="randn", scale=2.0).cuda()
    g = seeded(63, *wshape, dtype=dtype, kind="randn").cuda()
    w1, a1, w2, a2 = (t.clone().requires_grad_() for t in (w, alpha, w, alpha))
    e1, e2 = element(w1, a1, mode), w_tilde(w2, a2, mode)
    assert type(e1.grad_fn).__name__ != type(e2.grad_fn).__name__  # the fused operator ran
    assert torch.equal(e1, e2)
    # Gradients in 64 bits: each differs by roundings of the element's own type.
    w64, a64 = (t.double().requires_grad_() for t in (w, alpha))
    ref = torch.autograd.grad(w_tilde(w64, a64, mode), (w64, a64), g.double())
    for got, want in zip(torch.autograd.grad(e1, (w1, a1), g), ref):
        assert got.shape == want.shape and normwise_error(got.cpu().numpy(), want.cpu().numpy()) <= TOL[dtype]


def test_element_other_forms():
    """Forms the operator does not take run the torch operations; a graph of the backward is kept."""
    w = seeded(64, 3, 2, 3, 3).cuda()
    for alpha, mode in ((seeded(65, 1).cuda(), "sum"), (seeded(65, 3, 2, dtype=torch.float64).cuda(), "sum"), (seeded(65, 3).cuda(), "mean")):
        assert torch.equal(element(w, alpha, mode), w_tilde(w, alpha, mode))
    wp = w.permute(0, 1, 3, 2)
    alpha = seeded(66, 3, 2).cuda()
    assert torch.equal(element(wp, alpha), w_tilde(wp, alpha))
    a1, a2, w1, w2 = (t.double().clone().requires_grad_() for t in (alpha, alpha, w, w))
    seconds = []
    for f, a, v in ((element, a1, w1), (w_tilde, a2, w2)):
        first = torch.autograd.grad(f(v, a).square().sum(), (v, a), create_graph=True)
        seconds.append(torch.autograd.grad(sum(t.square().sum() for t in first), (v, a)))
    for got, want in zip(*seconds):
        assert normwise_error(got.cpu().numpy(), want.cpu().numpy()) <= 1e-12


def test_element_refuses_what_the_torch_operations_refuse():
    """Identity alphas whose strides cannot be viewed as one value per channel."""
    w, alpha = seeded(69, 6, 1, 3, 3).cuda(), seeded(70, 2, 3).cuda()
    for f in (element, w_tilde):
        assert f(w, alpha, "identity").shape == w.shape
        with pytest.raises(RuntimeError, match="view"):
            f(w, alpha.t(), "identity")


def test_element_keeps_strided_inputs_in_the_graph():
    """Second gradients of an element and alpha that are strided views reach both."""
    w, alpha = seeded(67, 3, 2, 5, 3, dtype=torch.float64).cuda(), seeded(68, 2, 3, dtype=torch.float64).cuda()
    seconds = []
    for f in (element, w_tilde):
        v, a = w.clone().requires_grad_(), alpha.clone().requires_grad_()
        vt, at = v.permute(0, 1, 3, 2), a.t()
        first = torch.autograd.grad(f(vt, at).square().sum(), (vt, at), create_graph=True)
        seconds.append(torch.autograd.grad(sum(t.square().sum() for t in first), (v, a)))
    for got, want in zip(*seconds):
        assert normwise_error(got.cpu().numpy(), want.cpu().numpy()) <= 1e-12


def _gradients(x, w, alpha, g):
    xd, wd, ad = (t.cuda().requires_grad_() for t in (x, w, alpha))
    torch.ops.morphocore.smorph(xd, wd, ad, O.MERGES["sum"]).backward(g.cuda())
    return [t.grad.cpu().numpy() for t in (xd, wd, ad)]


BIG = 1e4  # a float32 partial sum of this size loses 6e-4 of terms around 1; a double one 1e-12
ONCE = 2.0 ** -22  # two results, each the double sum rounded once


@pytest.mark.parametrize("KH,KW", [(9, 9), (6, 6)])
def test_float32_grad_input_of_many_slices_is_rounded_once(KH, KW):
    """Output channels in equal pairs with opposite large gradients cancel, whichever workgroups sum them:
    grad_input is that of the two channels left, whose gradients are small."""
    B, Cin, Cout, H, W = 1, 2, 258, 12, 40
    x = seeded(81, B, Cin, H, W, kind="randn")
    w = seeded(82, Cout, Cin, KH, KW, kind="randn", scale=0.2)
    alpha = seeded(83, Cout, Cin, kind="randn", scale=2.0)
    large = BIG * seeded(84, B, Cout - 2, H, W, kind="randn")
    w[1:-2:2], alpha[1:-2:2], large[:, 1::2] = w[:-2:2], alpha[:-2:2], -large[:, ::2]
    small = seeded(85, B, 2, H, W, kind="randn")
    got = _gradients(x, w, alpha, torch.cat([large, small], 1))[0]
    want = _gradients(x, w, alpha, torch.cat([torch.zeros_like(large), small], 1))[0]
    assert normwise_error(got, want) <= ONCE


@pytest.mark.parametrize("KH,KW", [(9, 9), (5, 3)])
def test_float32_slots_of_many_tiles_are_rounded_once(KH, KW):
    """Rows that see the same windows, in several tiles of one partial slot, with opposite large gradients
    cancel: grad_weight and grad_alpha are those of the row between them."""
    B, Cin, Cout, H, W = 128, 4, 1, 64, 40
    x = seeded(86, B, Cin, 1, W, kind="randn").expand(B, Cin, H, W).contiguous()
    w = seeded(87, Cout, Cin, KH, KW, kind="randn", scale=0.2)
    alpha = seeded(88, Cout, Cin, kind="randn", scale=2.0)
    small, large = torch.zeros(B, Cout, H, W), torch.zeros(B, Cout, H, W)
    small[:, :, 38] = seeded(89, B, Cout, W, kind="randn")
    large[:, :, 33] = BIG * seeded(90, B, Cout, W, kind="randn")
    large[:, :, 46] = -large[:, :, 33]
    for got, want in list(zip(_gradients(x, w, alpha, small + large), _gradients(x, w, alpha, small)))[1:]:
        assert normwise_error(got, want) <= ONCE


@pytest.mark.parametrize("merge", ["sum", "max", "identity", "smooth"])
def test_float32_batches_whose_sums_exceed_the_workspace_bound(merge):
    """Three batch elements of 544 MB of double grad_input sums each are taken one after the other: each gets the
    gradients it has alone, and the element those summed over the batch."""
    B, C, H, W, KH, KW = 3, 1, 8192, 8300, 1, 3
    gen = torch.Generator(device="cuda").manual_seed(95)
    x, g = (torch.randn(B, C, H, W, device="cuda", generator=gen) for _ in range(2))
    w = seeded(96, C, C, KH, KW, kind="randn", scale=0.2).cuda()
    alpha, beta = seeded(97, C, C, kind="randn").cuda(), seeded(98, C, kind="randn").cuda()

    def grads(xs, gs):
        leaves = [t.clone().requires_grad_() for t in (xs, w, alpha) + ((beta,) if merge == "smooth" else ())]
        out = torch.ops.morphocore.smorph_scm(*leaves) if merge == "smooth" else torch.ops.morphocore.smorph(*leaves, O.MERGES[merge])
        return torch.autograd.grad(out, leaves, gs)

    whole = grads(x, g)
    alone = [grads(x[b:b + 1], g[b:b + 1]) for b in range(B)]
    for b in range(B):
        assert torch.equal(whole[0][b], alone[b][0][0])
    for k in range(1, len(whole)):
        want = sum(a[k].double() for a in alone)
        assert normwise_error(whole[k].cpu().numpy(), want.cpu().numpy()) <= 1e-6
