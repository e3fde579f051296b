"""Residual add, RMS norm, depthwise convolution and projection of few images in one kernel against the kernels it stands for: grids smaller
than a patch, ragged patches, one and many column tiles, several images, both widths."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,h,w,C,N,full", [(1, 14, 14, 192, 640, True), (1, 1, 1, 192, 128, False), (2, 3, 17, 192, 256, True),
                                            (1, 14, 14, 384, 1280, True), (3, 5, 8, 384, 128, False), (1, 33, 9, 384, 128, True)])
def test_against_separate_kernels(B, h, w, C, N, full):
    announce(f"norm, convolution and projection B{B} {h}x{w} C{C} N{N}")
    gen = torch.Generator().manual_seed(7 * h + w)
    rows = B * h * w
    r = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    x, res, wt = r(rows, C).bfloat16().cuda(), r(rows, C).bfloat16().cuda() if full else None, (r(N, C) * C ** -0.5).bfloat16().cuda()
    nw, taps = (torch.rand(C, generator=gen) + 0.5).cuda(), (r(C, 9) / 3).cuda()
    cb, b = (r(C).cuda(), r(N).bfloat16().cuda()) if full else (None, None)
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    assert lib.vig_norm_dwconv3x3_linear_preferred(B, h, w, C, N)
    total, conv, y = (torch.full((rows, n), float("nan"), dtype=torch.bfloat16, device="cuda") for n in (C, C, N))
    assert lib.vig_norm_dwconv3x3_linear_fwd(p(x), p(res), p(nw), p(taps), p(cb), p(wt), p(b), p(total) if full else None, p(conv), p(y), B, h, w,
                                             C, N, 1e-5, full, st) == _lib.VIG_OK
    normed, total2, conv2, y2 = (torch.empty(rows, n, dtype=torch.bfloat16, device="cuda") for n in (C, C, C, N))
    assert lib.vig_rmsnorm_fwd(p(x), p(res), p(nw), p(normed), p(total2), rows, C, 1e-5, 1, 1, st) == _lib.VIG_OK
    assert lib.vig_dwconv3x3_fwd(p(normed), p(taps), p(cb), p(conv2), B, h, w, C, full, 1, st) == _lib.VIG_OK
    if full:
        assert torch.equal(total, total2)
    assert lib.vig_linear_fwd(p(conv2), C, p(wt), p(b), p(y2), N, rows, N, C, st) == _lib.VIG_OK
    assert torch.equal(conv, conv2) and torch.equal(y, y2)  # the same sums in the same order


def test_refused():
    t = [torch.zeros(4096, 384, dtype=torch.bfloat16, device="cuda") for _ in range(6)]
    f, lib, st = torch.ones(384 * 9, device="cuda"), _lib.load(), torch.cuda.current_stream().cuda_stream
    call = lambda x, res, s, c, y, B, C, N: lib.vig_norm_dwconv3x3_linear_fwd(  # noqa: E731
        x.data_ptr(), res.data_ptr(), f.data_ptr(), f.data_ptr(), None, t[5].data_ptr(), None, s.data_ptr(), c.data_ptr(), y.data_ptr(), B, 4, 8, C,
        N, 1e-5, 0, st)
    a, b, s, c, y = t[:5]
    assert call(a, b, s, c, y, 1, 384, 128) == _lib.VIG_OK
    for outs in ((a, c, y), (s, a, y), (s, c, a), (b, c, y), (s, b, y), (s, c, b), (s, s, y), (s, c, c), (s, c, s), (t[5], c, y)):
        assert call(a, b, *outs, 1, 384, 128) == _lib.VIG_EINVAL
    assert call(a, b, s, c, y, 1, 256, 128) == _lib.VIG_ENOTSUP  # another width
    assert call(a, b, s, c, y, 1, 384, 192) == _lib.VIG_ENOTSUP  # half a column tile
    assert call(a, b, s, c, y, 128, 384, 384) == _lib.VIG_ENOTSUP  # many images
