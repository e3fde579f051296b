"""The bf16 product either side of the line between its 64 x 64 and 128 x 128 tiles (512 of the small ones), with rows, columns and
contractions that end inside a tile or a stage, against fp64."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1600, 1280, 384), (1664, 1280, 384), (2049, 1288, 32), (4097, 520, 96), (1700, 2568, 768), (33000, 72, 64),
                                   (900, 4096, 352)])
@pytest.mark.parametrize("bias", [False, True])
def test_product(M, N, K, bias):
    announce(f"product tiles M{M} N{N} K{K} bias={bias}")
    gen = torch.Generator().manual_seed(M)
    x, w, b = (torch.randn(s, generator=gen).bfloat16().cuda() for s in ((M, K), (N, K), (N,)))
    y = torch.full((M, N + 8), 3.0, dtype=torch.bfloat16, device="cuda")
    lib = _lib.load()
    assert lib.vig_linear_preferred(M, N, K)
    assert lib.vig_linear_fwd(x.data_ptr(), K, w.data_ptr(), b.data_ptr() if bias else None, y.data_ptr(), N + 8, M, N, K,
                              torch.cuda.current_stream().cuda_stream) == _lib.VIG_OK
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    # the one rounding to bf16, and an fp32 rounding for every 16 contraction steps
    bound = want.abs() * 2.0 ** -8 + (K / 16 + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs()) + 1e-30
    assert ((y[:, :N].double() - want).abs() <= bound).all() and (y[:, N:] == 3.0).all()
