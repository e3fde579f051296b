"""Residual add, RMS norm and depthwise convolution in one kernel against the two kernels it stands for: single cells, rows
narrower and wider than a workgroup's cells, images next to each other, both widths, with and without the options; walks of a few
rows with a short last band, and of all rows."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,h,w,C,full", [(1, 1, 1, 192, True), (1, 14, 14, 192, True), (2, 14, 14, 384, False), (3, 5, 15, 384, True),
                                          (1, 3, 17, 192, False), (1, 4, 29, 384, True), (1, 2, 64, 192, True),
                                          (100, 13, 14, 384, True), (64, 13, 27, 192, False), (250, 14, 14, 384, True)])
def test_against_two_kernels(B, h, w, C, full):
    announce(f"norm and convolution {B}x{h}x{w}x{C} options {full}")
    gen = torch.Generator().manual_seed(h * w)
    x, res = (torch.randn(B, h * w, C, generator=gen).bfloat16().cuda() for _ in range(2))
    wt, bias, nw = (torch.randn(C, 9, generator=gen) / 3).cuda(), torch.randn(C, generator=gen).cuda(), (torch.rand(C, generator=gen) + 0.5).cuda()
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    p = lambda t: t.data_ptr() if t is not None and (full or t is not res and t is not bias) else None  # noqa: E731
    assert lib.vig_norm_dwconv3x3_preferred(B, h, w, C)
    total, y = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    assert lib.vig_norm_dwconv3x3_fwd(p(x), p(res), p(nw), p(wt), p(bias), total.data_ptr() if full else None, p(y), B, h, w, C, 1e-5,
                                      int(full), st) == _lib.VIG_OK
    normed, sum2, want = (torch.empty_like(x) for _ in range(3))
    assert lib.vig_rmsnorm_fwd(p(x), p(res), p(nw), p(normed), sum2.data_ptr() if full else None, B * h * w, C, 1e-5, int(full), 1, st) == _lib.VIG_OK
    assert lib.vig_dwconv3x3_fwd(p(normed), p(wt), p(bias), p(want), B, h, w, C, int(full), 1, st) == _lib.VIG_OK
    assert not full or torch.equal(total, sum2)
    assert torch.equal(y, want)  # the same sums in the same order


def test_refused():
    t, f, lib, st = torch.zeros(64, 192, dtype=torch.bfloat16, device="cuda"), torch.ones(192 * 9, device="cuda"), _lib.load(), torch.cuda.current_stream().cuda_stream
    out, total = torch.zeros_like(t), torch.zeros_like(t)
    call = lambda s, y, h, w, C: lib.vig_norm_dwconv3x3_fwd(t.data_ptr(), None, f.data_ptr(), f.data_ptr(), None, s, y, 1, h, w, C, 1e-5, 0, st)  # noqa: E731
    assert call(total.data_ptr(), out.data_ptr(), 8, 8, 192) == _lib.VIG_OK
    assert call(t.data_ptr(), out.data_ptr(), 8, 8, 192) == _lib.VIG_EINVAL and call(None, t.data_ptr(), 8, 8, 192) == _lib.VIG_EINVAL
    assert call(None, out.data_ptr(), 8, 8, 64) == _lib.VIG_ENOTSUP and call(None, out.data_ptr(), 1 << 20, 1 << 10, 192) == _lib.VIG_ENOTSUP
