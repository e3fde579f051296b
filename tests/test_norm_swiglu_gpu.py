"""Residual add, RMS norm and SwiGLU layer of few rows in one kernel against the two kernels it stands for: one row, ragged row tiles, one
and many column tiles, both widths."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,K,I", [(1, 192, 32), (49, 192, 512), (196, 192, 512), (33, 384, 1024), (196, 384, 1024), (256, 384, 1024), (2048, 192, 128)])
def test_against_two_kernels(rows, K, I):
    announce(f"norm and SwiGLU rows{rows} K{K} I{I}")
    gen = torch.Generator().manual_seed(rows)
    x, res = (torch.randn(rows, K, generator=gen).bfloat16().cuda() for _ in range(2))
    w = (torch.randn(2 * I, K, generator=gen) * K ** -0.5).bfloat16().cuda()
    nw = (torch.rand(K, generator=gen) + 0.5).cuda()
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    assert lib.vig_norm_swiglu_preferred(rows, K, I)
    total, y = torch.full_like(x, float("nan")), torch.full((rows, I), float("nan"), dtype=x.dtype, device="cuda")
    assert lib.vig_norm_swiglu_fwd(*(t.data_ptr() for t in (x, res, nw, w, total, y)), rows, K, I, 1e-5, st) == _lib.VIG_OK
    normed, sum2, want = torch.empty_like(x), torch.empty_like(x), torch.empty_like(y)
    assert lib.vig_rmsnorm_fwd(x.data_ptr(), res.data_ptr(), nw.data_ptr(), normed.data_ptr(), sum2.data_ptr(), rows, K, 1e-5, 0, 1, st) == _lib.VIG_OK
    assert lib.vig_linear_swiglu_fwd(normed.data_ptr(), w.data_ptr(), want.data_ptr(), rows, K, I, 1, st) == _lib.VIG_OK
    assert torch.equal(total, sum2)
    assert torch.equal(y, want)  # the same sums in the same order


def test_refused():
    x, res, w, out, total = (torch.zeros(2048, 384, dtype=torch.bfloat16, device="cuda") for _ in range(5))
    f, lib, st = torch.ones(384, device="cuda"), _lib.load(), torch.cuda.current_stream().cuda_stream
    call = lambda s, y, rows, K, I: lib.vig_norm_swiglu_fwd(x.data_ptr(), res.data_ptr(), f.data_ptr(), w.data_ptr(), s.data_ptr(), y.data_ptr(),  # noqa: E731
                                                            rows, K, I, 1e-5, st)
    assert call(total, out, 32, 384, 32) == _lib.VIG_OK
    for s, y in ((x, out), (res, out), (total, x), (total, res), (total, total)):  # an output over an input or the other output
        assert call(s, y, 32, 384, 32) == _lib.VIG_EINVAL
    assert call(total, out, 2048, 384, 1024) == _lib.VIG_ENOTSUP  # many rows
    assert call(total, out, 32, 256, 32) == _lib.VIG_ENOTSUP  # another width
