"""The convolutions of the patch embedding in training: the kernels' values against fp64 on the rounded inputs, torch's own gradients, the calls that stay with
torch, and a graph of the gradients."""
import pytest
import torch
import torch.nn.functional as F

from vig_amd import _ext

from .util import announce

pytestmark = pytest.mark.gpu


def _case(B, Cin, Cout, k, H, W, seed=0):
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(B, Cin, H, W, generator=g).cuda(), torch.randn(Cout, Cin, k, k, generator=g).cuda() / (Cin * k * k) ** 0.5
    if k == 3:
        x = x.contiguous(memory_format=torch.channels_last)
    return x, w.contiguous(memory_format=torch.channels_last).requires_grad_()


def _amp(fn, *a):
    with torch.autocast("cuda", dtype=torch.bfloat16):
        return fn(*a)


@pytest.mark.parametrize("B,Cin,Cout,k,H,W", [(1, 3, 64, 9, 7, 8), (2, 3, 96, 9, 40, 24), (3, 3, 192, 9, 33, 264), (1, 3, 384, 9, 64, 64), (1, 32, 8, 3, 1, 1),
                                              (2, 96, 192, 3, 5, 7), (9, 192, 384, 3, 28, 28)])
def test_values_and_gradients(B, Cin, Cout, k, H, W):
    announce(f"stem conv B{B} {Cin}->{Cout} {k}x{k} of {H}x{W}")
    x, w = _case(B, Cin, Cout, k, H, W)
    x.requires_grad_(k == 3)
    s = 8 if k == 9 else 2
    y = _amp(_ext.calls().stem_conv, x, w, s)
    want = F.conv2d(x.detach().bfloat16().double(), w.detach().bfloat16().double(), None, s, 1)
    assert y.dtype == torch.bfloat16 and y.shape == want.shape and y.permute(0, 2, 3, 1).is_contiguous()
    assert ((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()  # the stored value's rounding; fp32 sums of up to 1728 terms
    dy = torch.randn(y.shape, device="cuda").bfloat16().contiguous(memory_format=torch.channels_last)
    ins = [w] + [x] * (k == 3)
    other = _amp(F.conv2d, x, w, None, s, 1)
    for a, b in zip(torch.autograd.grad(y, ins, dy), torch.autograd.grad(other, ins, dy)):
        assert a.dtype == b.dtype and (a - b).norm() <= 1e-2 * b.norm()  # torch's operator for both (its sums need not have one order)


@pytest.mark.parametrize("kw,W", [(9, 40), (9, 264), (3, 24), (16, 40)])
def test_a_pixel_that_is_not_finite(kw, W):
    """One in each image, at every column and a third of the rows: it reaches the windows that hold it and no other."""
    announce(f"stem conv, pixels that are not finite, {kw} columns of {W}")
    g = torch.Generator().manual_seed(kw)
    x, w = torch.randn(W, 3, 25, W, generator=g).bfloat16(), (torch.randn(64, 3, 9, kw, generator=g) / 9).bfloat16()
    at = torch.arange(W)
    x[at, at % 3, at % 25, at] = torch.tensor([float("inf"), float("-inf"), float("nan")], dtype=torch.bfloat16)[at % 3]
    want = F.conv2d(x.float(), w.float(), None, 8, 1)
    got = _amp(_ext.calls().stem_conv, x.cuda(), w.float().cuda().contiguous(memory_format=torch.channels_last), 8).float().cpu()
    assert 0 < want.isfinite().float().mean() < 1 and torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    held = want.isfinite()
    assert torch.equal(got[want.isinf()], want[want.isinf()]) and ((got - want)[held].abs() <= 2.0 ** -8 * want[held].abs() + 1e-5).all()


def test_stays_with_torch():
    announce("stem conv: calls that stay with torch")
    take = _ext.calls().stem_conv
    x, w = _case(2, 3, 96, 9, 40, 24)
    assert take(x, w, 8) is None  # fp32
    assert _amp(take, x, w, 8) is not None
    with torch.autocast("cuda", dtype=torch.float16):
        assert take(x, w, 8) is None
    assert _amp(take, x.contiguous(memory_format=torch.channels_last), w, 8) is None and _amp(take, x[:, :, :, :20], w, 8) is None
    assert _amp(take, x, w[:40], 8) is None and _amp(take, x, w, 4) is None and _amp(take, x.double(), w, 8) is None
    x, w = _case(2, 32, 64, 3, 6, 6)
    assert _amp(take, x, w, 2) is not None
    assert _amp(take, x.contiguous(), w, 2) is None and _amp(take, x[:, :24], w[:, :24], 2) is None and _amp(take, x, w.contiguous(), 2) is None


def test_graph_of_the_gradients():
    announce("stem conv: second derivatives")
    x, w = _case(1, 32, 64, 3, 6, 6, 1)
    x.requires_grad_()
    d = torch.randn(1, 64, 3, 3, device="cuda").bfloat16()

    def second(y):
        first = torch.autograd.grad(y, [x, w], d, create_graph=True)
        return torch.autograd.grad(sum(t.square().sum() for t in first), [x, w])

    for a, b in zip(second(_amp(_ext.calls().stem_conv, x, w, 2)), second(_amp(F.conv2d, x, w, None, 2, 1))):
        assert (a - b).norm() <= 2e-2 * b.norm()
