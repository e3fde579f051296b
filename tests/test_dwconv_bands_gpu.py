"""Backward of the depthwise convolution where its bands can go wrong: few images (short bands, a workgroup each), bands of part of a row,
channel tails, weights that start off a 16-byte boundary, the smallest workspace; against fp64."""
import pytest
import torch
import torch.nn.functional as F

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("least", [False, True])
@pytest.mark.parametrize("dtype,eps", [(torch.float32, 2.0 ** -20), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("B,h,w,C", [(1, 1, 1, 8), (1, 3, 5, 72), (2, 14, 14, 64), (1, 33, 40, 192), (1, 70, 64, 8), (1, 5, 100, 72), (90, 14, 14, 384)])
def test_gradients(B, h, w, C, dtype, eps, least):
    announce(f"depthwise gradients B{B} {h}x{w} C{C} {dtype} least workspace {least}")
    gen = torch.Generator().manual_seed(h * w)
    x, dy = (torch.randn(B, h * w, C, generator=gen).to(dtype).cuda() for _ in range(2))
    store = torch.randn(C * 9 + 1, generator=gen).cuda()
    wt = store[1:] if least else store[:-1]  # (off the boundary, and on it)
    lib, code = _lib.load(), int(dtype == torch.bfloat16)
    size = B * 4 * C * 10 * 4 if least else lib.vig_dwconv3x3_bwd_weight_workspace(B, C)
    ws = torch.full((size + 512,), 77, dtype=torch.uint8, device="cuda")
    dx, dw = torch.empty_like(x), torch.empty(C * 10, device="cuda")
    args = (x.data_ptr(), dy.data_ptr(), None, wt.data_ptr(), dx.data_ptr(), dw.data_ptr(), ws.data_ptr())
    tail = (B, h, w, C, code, torch.cuda.current_stream().cuda_stream)
    assert lib.vig_dwconv3x3_bwd(*args, B * 4 * C * 10 * 4 - 4, *tail) == _lib.VIG_ENOSPC
    assert lib.vig_dwconv3x3_bwd(*args, size, *tail) == _lib.VIG_OK and (ws[size:] == 77).all()
    grid = lambda t: t.double().cpu().transpose(1, 2).reshape(B, C, h, w)  # noqa: E731
    x64, w64, b64 = grid(x).requires_grad_(), wt.double().cpu().reshape(C, 1, 3, 3).requires_grad_(), torch.zeros(C, dtype=torch.float64).requires_grad_()
    F.conv2d(x64, w64, b64, padding=1, groups=C).backward(grid(dy))
    assert ((grid(dx) - x64.grad).abs() <= eps * x64.grad.abs().max()).all()
    got, n = dw.double().cpu(), B * h * w  # fp32 sums of n products in any order: roundings that grow with the root of n, 5 sigma of terms
    for part, want in ((got[:C * 9], w64.grad.reshape(-1)), (got[C * 9:], b64.grad)):
        assert (part - want).abs().max() <= 2.0 ** -21 * 5 * n ** 0.5 + 2.0 ** -21 * want.abs().max()
