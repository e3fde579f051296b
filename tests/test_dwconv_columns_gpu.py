"""The depthwise convolution's two forms where they can go wrong: single rows and columns, bands of part of an image, channel tails, columns
that end inside a workgroup, both sides of the line between the forms; against fp64."""
import pytest
import torch
import torch.nn.functional as F

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,eps", [(torch.float32, 2.0 ** -20), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("silu,keep,biased", [(0, False, False), (1, False, True), (1, True, True)])
@pytest.mark.parametrize("B,h,w,C", [(1, 1, 1, 8), (2, 1, 9, 72), (2, 9, 1, 64), (1, 5, 40, 72), (1, 70, 41, 8), (3, 14, 14, 192),
                                     (669, 14, 14, 64), (670, 14, 14, 64)])  # 149 856 and 150 080 columns of quads
def test_forms(B, h, w, C, silu, keep, biased, dtype, eps):
    announce(f"depthwise forward B{B} {h}x{w} C{C} {dtype} silu {silu} pre {keep}")
    gen = torch.Generator().manual_seed(h * w + C)
    x = torch.randn(B, h * w, C, generator=gen).to(dtype).cuda()
    wt, bias = torch.randn(C * 9, generator=gen).cuda(), torch.randn(C, generator=gen).cuda()
    y, pre = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    rc = _lib.load().vig_dwconv3x3_fwd_pre(x.data_ptr(), wt.data_ptr(), bias.data_ptr() if biased else None, y.data_ptr(),
                                           pre.data_ptr() if keep else None, B, h, w, C, silu, int(dtype == torch.bfloat16),
                                           torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.VIG_OK
    grid = lambda t: t.double().cpu().transpose(1, 2).reshape(B, C, h, w)  # noqa: E731
    w64, b64 = wt.double().cpu().reshape(C, 1, 3, 3), bias.double().cpu() if biased else None
    want = F.conv2d(grid(x), w64, b64, padding=1, groups=C)
    # nine products and a bias in fp32, then one rounding to the type: relative to the sum of magnitudes
    size = F.conv2d(grid(x).abs(), w64.abs(), b64.abs() if biased else None, padding=1, groups=C)
    if keep:
        assert ((grid(pre) - want).abs() <= eps * size).all()
        want = grid(pre)  # (the activation reads the stored value)
    if silu:
        want = want * torch.sigmoid(want)  # (its slope stays below 1.1)
    assert ((grid(y) - want).abs() <= 1.2 * eps * size).all()


@pytest.mark.parametrize("dtype,eps", [(torch.float32, 2.0 ** -20), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("B,h,w,C", [(390, 7, 14, 64), (391, 7, 14, 64), (585, 9, 14, 64), (586, 16, 14, 64), (586, 17, 14, 64)])
def test_bands_that_fit_a_round(B, h, w, C, dtype, eps):
    """Both sides of the lines between three, two and one band: 87 360 and 87 584 columns of quads, 131 040 and 131 264."""
    test_forms(B, h, w, C, 1, True, True, dtype, eps)
