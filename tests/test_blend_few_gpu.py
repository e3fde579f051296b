"""The mixer's epilogue and o_proj of few rows against fp64: one row, ragged row tiles, tokens of several images, pitched gate rows, both
widths; the same inputs as part of a batch that takes the kernel of many rows give the same values but for the order of the sums."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,H,silu,pitch", [(1, 1, 3, 0, 0), (1, 196, 3, 0, 64), (3, 49, 6, 1, 0), (2, 130, 6, 0, 128), (33, 31, 3, 1, 0)])
def test_against_fp64(B, L, H, silu, pitch):
    announce(f"blend and projection B{B} L{L} H{H} silu{silu} pitch{pitch}")
    C, gen = 64 * H, torch.Generator().manual_seed(L)
    o, loc = torch.randn(B, H, L, 64, generator=gen).bfloat16().cuda(), torch.randn(B, L, C, generator=gen).bfloat16().cuda()
    wide = torch.randn(B, L, C + pitch, generator=gen).bfloat16().cuda()
    g, w = wide[..., pitch:], (torch.randn(C, C, generator=gen) * C ** -0.5).bfloat16().cuda()
    wg, wl = ((torch.rand(64, generator=gen) + 0.5).cuda() for _ in range(2))
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream

    def run(o, loc, g, B):
        out = torch.full((B, L, C), float("nan"), dtype=o.dtype, device="cuda")
        assert lib.vig_locality_blend_linear_fwd(o.data_ptr(), loc.data_ptr(), g.data_ptr(), wg.data_ptr(), wl.data_ptr(), w.data_ptr(), out.data_ptr(),
                                                 B, H, L, 64, C, C + pitch, 1e-5, silu, 1, st) == _lib.VIG_OK
        return out

    got = run(o, loc, g, B)
    norm = lambda x, weight: x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * weight.double()  # noqa: E731
    s = torch.sigmoid(g.double().reshape(B, L, H, 64))
    y = norm(o.double().transpose(1, 2), wg) * s + norm(loc.double().reshape(B, L, H, 64), wl) * (1 - s)
    y = (torch.nn.functional.silu(y) if silu else y).reshape(B, L, C)
    want = y @ w.double().t()
    # y rounded to bf16 once (2^-9 of each term, independent: 8 sigma of the root of the sum of squares), the result once
    bound = 8 * 2.0 ** -9 * (y.pow(2) @ w.double().pow(2).t()).sqrt() + 2.0 ** -8 * want.abs() + 1e-5
    assert ((got.double() - want).abs() <= bound).all()
    many = 1 + 6000 // (B * L)  # copies of the batch, past the row count of the kernel of few rows
    ref = run(o.repeat(many, 1, 1, 1), loc.repeat(many, 1, 1), wide.repeat(many, 1, 1)[..., pitch:], many * B)[:B]
    assert (got != ref).float().mean() < 0.02 and (got.float() - ref.float()).abs().max() <= 2.0 ** -7 * ref.float().abs().max()


def test_result_over_an_input():
    gen = torch.Generator().manual_seed(1)
    o, loc, g = torch.randn(1, 3, 196, 64, generator=gen).bfloat16().cuda(), *(torch.randn(1, 196, 192, generator=gen).bfloat16().cuda() for _ in range(2))
    w, n = torch.randn(192, 192, generator=gen).bfloat16().cuda(), torch.ones(64, device="cuda")
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    call = lambda out, x, y: lib.vig_locality_blend_linear_fwd(o.data_ptr(), x.data_ptr(), y.data_ptr(), n.data_ptr(), n.data_ptr(), w.data_ptr(),  # noqa: E731
                                                               out.data_ptr(), 1, 3, 196, 64, 192, 192, 1e-5, 0, 1, st)
    want, over_loc, over_g = torch.empty_like(loc), loc.clone(), g.clone()
    assert call(want, loc, g) == call(over_loc, over_loc, g) == call(over_g, loc, over_g) == _lib.VIG_OK
    for got in (over_loc, over_g):  # the kernel of whole rows: sums in another order, an ulp of bf16 now and then
        assert (got != want).float().mean() < 0.02 and (got.float() - want.float()).abs().max() <= 2.0 ** -7 * want.float().abs().max()
