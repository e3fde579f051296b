"""The middle of a block of few rows in one kernel (blend, o_proj, residual add, norm, SwiGLU layer) against the kernels it stands for: one row, ragged
row tiles, one and many column tiles, several images, rows of a wider gate matrix."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


def _case(B, L, I, ld, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    M = B * L
    bf = [t.bfloat16().cuda() for t in (r(B, 3, L, 64), r(M, 192), r(M, ld), r(192, 192) / 14, r(M, 192), r(2 * I, 192) / 14)]
    f = [(torch.rand(n, generator=g) + 0.5).cuda() for n in (64, 64, 192)]
    return bf, f


@pytest.mark.parametrize("B,L,I,ld,act", [(1, 1, 64, 192, 1), (1, 196, 512, 640, 1), (3, 33, 512, 208, 0), (2, 16, 64, 192, 0), (1, 512, 512, 640, 1)])
def test_against_separate_kernels(B, L, I, ld, act):
    announce(f"blend, o_proj, norm and SwiGLU B{B} L{L} I{I} pitch{ld}")
    M, lib, st = B * L, _lib.load(), torch.cuda.current_stream().cuda_stream
    (o, loc, glin, wo, res, w), (wg, wl, nw) = _case(B, L, I, ld, L + I)
    p = lambda t: t.data_ptr()  # noqa: E731
    assert lib.vig_locality_blend_swiglu_preferred(M, 192, I)
    new = lambda n: torch.full((M, n), float("nan"), dtype=torch.bfloat16, device="cuda")  # noqa: E731
    total, y, a, total2, y2 = new(192), new(I), new(192), new(192), new(I)
    assert lib.vig_locality_blend_swiglu_fwd(p(o), p(loc), p(glin), p(wg), p(wl), p(wo), p(res), p(nw), p(w), p(total), p(y), B, 3, L, 64, 192, I, ld,
                                             1e-5, act, 1e-6, st) == _lib.VIG_OK
    assert lib.vig_locality_blend_linear_fwd(p(o), p(loc), p(glin), p(wg), p(wl), p(wo), p(a), B, 3, L, 64, 192, ld, 1e-5, act, 1, st) == _lib.VIG_OK
    assert lib.vig_norm_swiglu_fwd(p(a), p(res), p(nw), p(w), p(total2), p(y2), M, 192, I, 1e-6, st) == _lib.VIG_OK
    assert torch.equal(total, total2) and torch.equal(y, y2)  # the same sums in the same order


def test_refused():
    (o, loc, glin, wo, res, w), (wg, wl, nw) = _case(1, 64, 64, 192, 0)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    total, y = torch.empty_like(loc), torch.empty(64, 192, dtype=torch.bfloat16, device="cuda")

    def call(total=total, y=y, H=3, L=64, Dv=64, C=192, I=64, ld=192):
        return lib.vig_locality_blend_swiglu_fwd(*(t.data_ptr() for t in (o, loc, glin, wg, wl, wo, res, nw, w, total, y)), 1, H, L, Dv, C, I, ld, 1e-5,
                                                 1, 1e-6, st)

    assert call() == _lib.VIG_OK
    for t in (o, loc, glin, wo, res, w):  # an output over an input
        assert call(total=t) == _lib.VIG_EINVAL and call(y=t) == _lib.VIG_EINVAL
    assert call(y=total) == _lib.VIG_EINVAL and call(ld=184) == _lib.VIG_EINVAL and call(ld=196) == _lib.VIG_EINVAL
    assert call(I=32) == _lib.VIG_ENOTSUP and call(H=6, C=384) == _lib.VIG_ENOTSUP and call(H=6, Dv=32) == _lib.VIG_ENOTSUP
    assert call(L=5000) == _lib.VIG_ENOTSUP  # many rows
