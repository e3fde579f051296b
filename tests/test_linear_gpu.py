"""The linear layers with their weights in registers, and SwiGLU of a layer in its three forms, where they can go wrong: against
float64 sums of the same bf16 values."""
import pytest
import torch

import vig_amd
from vig_amd import _lib, ops

from .util import announce

pytestmark = pytest.mark.gpu


def _randn(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).bfloat16()


def _check(got, want64, ulps=1.0):
    """Within `ulps` bf16 roundings (2^-8 relative) and the fp32 sums' error, 1e-5 of the result's scale."""
    got = got.double().cpu()
    assert ((got - want64).abs() <= ulps * 2.0 ** -8 * want64.abs() + 1e-5 * want64.abs().max()).all()


# the first sizes of the rule; ragged token tiles; one, some and all of a workgroup's channel tiles, both contractions
@pytest.mark.parametrize("rows,N,K", [(16384, 64, 192), (16385, 320, 384), (20011, 704, 192), (16415, 1280, 384),
                                      (8192, 512, 192), (8209, 768, 192), (10752, 1536, 384), (10783, 2112, 384)])
def test_linear_in_registers(rows, N, K):
    announce(f"linear in registers rows{rows} N{N} K{K}")
    x, w, b = _randn((rows, K), 1), _randn((N, K), 2, K ** -0.5), _randn((N,), 3)
    assert vig_amd._lib.load().vig_linear_preferred(rows, N, K)
    for bias in (None, b):
        got = ops.linear(x.cuda(), w.cuda(), bias.cuda() if bias is not None else None)
        _check(got, torch.nn.functional.linear(x.double(), w.double(), bias.double() if bias is not None else None))


# both sides of the lines between the forms (256 result tiles, 1024 tokens), ragged tokens, channel tiles of part of a workgroup
@pytest.mark.parametrize("rows,K,I", [(1, 192, 32), (256, 384, 1024), (257, 384, 1024), (1024, 384, 1056), (1025, 384, 1056),
                                      (8192, 192, 32), (8193, 192, 32), (9000, 192, 160), (9001, 384, 288)])
def test_linear_swiglu_forms(rows, K, I):
    announce(f"linear_swiglu rows{rows} K{K} I{I}")
    x, w = _randn((rows, K), 4), _randn((2 * I, K), 5, K ** -0.5)
    xd, wd = x.cuda(), w.cuda()
    got = ops.linear_swiglu(xd, wd)
    z, y = (torch.full((rows, n), float("nan"), dtype=torch.bfloat16, device="cuda") for n in (2 * I, I))
    rc = _lib.load().vig_linear_swiglu_kept_fwd(xd.data_ptr(), wd.data_ptr(), z.data_ptr(), y.data_ptr(), rows, K, I, _lib.VIG_BF16,
                                                torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    want = x.double() @ w.double().t()
    _check(z, want)
    g, u = z.double().cpu().chunk(2, 1)
    _check(y, torch.nn.functional.silu(g) * u)  # of the values that were kept
    # a pre-activation that another summation order rounds the other way moves the product by an ulp of each factor
    g, u = want.chunk(2, 1)
    _check(got, torch.nn.functional.silu(g) * u, ulps=4.0)


# products with the weight's columns: the first size of the rule and below it, ragged tokens, channel tiles of part of a workgroup
@pytest.mark.parametrize("rows,N,K", [(1, 192, 64), (33, 384, 704), (16384, 384, 384), (16399, 192, 320)])
def test_linear_bwd_input(rows, N, K):
    announce(f"linear input gradient rows{rows} N{N} K{K}")
    dy, w = _randn((rows, N), 11), _randn((N, K), 12, N ** -0.5)
    lib, dyd, wd = _lib.load(), dy.cuda(), w.cuda()
    dx = torch.full((rows, K), float("nan"), dtype=torch.bfloat16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.vig_linear_bwd_input(dyd.data_ptr(), wd.data_ptr(), dx.data_ptr(), rows, N, K, _lib.VIG_BF16, stream) == 0
    _check(dx, dy.double() @ w.double())
    assert bool(lib.vig_linear_bwd_input_preferred(rows, N, K)) == (rows >= 16384)
    assert lib.vig_linear_bwd_input(dyd.data_ptr(), wd.data_ptr(), dx.data_ptr(), rows, N, 32, _lib.VIG_BF16, stream) != 0


@pytest.mark.parametrize("rows,K,I", [(1, 192, 32), (37, 384, 96), (2049, 192, 160), (9001, 384, 288)])
def test_linear_swiglu_bwd(rows, K, I):
    announce(f"linear_swiglu_bwd rows{rows} K{K} I{I}")
    dy, w, z = _randn((rows, K), 13), _randn((K, I), 14, K ** -0.5), _randn((rows, 2 * I), 15)
    lib, dyd, wd, zd = _lib.load(), dy.cuda(), w.cuda(), z.cuda()
    dz = torch.full((rows, 2 * I), float("nan"), dtype=torch.bfloat16, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.vig_linear_swiglu_bwd(dyd.data_ptr(), wd.data_ptr(), zd.data_ptr(), dz.data_ptr(), rows, K, I, _lib.VIG_BF16, stream) == 0
    d = dy.double() @ w.double()
    g, u = z.double().chunk(2, 1)
    s = torch.sigmoid(g)
    want = torch.cat((d * u * s * (1 + g * (1 - s)), d * g * s), 1)
    _check(dz, want, ulps=2.0)  # one rounding of the product's gradient, one of the result


# whole rows in one workgroup: ragged row tiles, the shortest contractions (stages short of the buffers) and longer ones
@pytest.mark.parametrize("rows,N,K", [(1, 192, 64), (129, 192, 128), (257, 192, 192), (4097, 192, 512), (16401, 192, 1024)])
def test_linear_norm(rows, N, K):
    announce(f"linear, residual add and norm rows{rows} N{N} K{K}")
    x, w, res = _randn((rows, K), 16), _randn((N, K), 17, K ** -0.5), _randn((rows, N), 18)
    nw = torch.rand(N, generator=torch.Generator().manual_seed(19)) + 0.5
    lib, dev = _lib.load(), [t.cuda() for t in (x, w, res, nw)]
    y, total = (torch.full((rows, N), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    rc = lib.vig_linear_norm_fwd(*(t.data_ptr() for t in (*dev, y, total)), rows, N, K, 1e-5, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    product = x.double() @ w.double().t()
    # one rounding of the product, one of the sum
    err = (total.double().cpu() - (product + res.double())).abs()
    assert (err <= 2.0 ** -8 * (product.abs() + (product + res.double()).abs()) + 1e-5 * product.abs().max()).all()
    s = total.double().cpu()
    _check(y, s / torch.sqrt((s * s).mean(1, keepdim=True) + 1e-5) * nw.double())  # of the sum that was stored
    assert bool(lib.vig_linear_norm_preferred(rows, N, K)) == (rows >= 16384)


# the mixer's epilogue with the output projection, blended rows kept: one token, ragged tiles, more tiles than workgroups
@pytest.mark.parametrize("B,L,H", [(1, 1, 3), (3, 37, 6), (1, 65, 3), (90, 197, 6)])
def test_blend_linear_kept(B, L, H):
    announce(f"blend_linear with the blended rows kept B{B} L{L} H{H}")
    C, ld = 64 * H, 64 * H + 64
    o, loc, w = _randn((B, H, L, 64), 20).cuda(), _randn((B, L, C), 21).cuda(), _randn((C, C), 22, C ** -0.5).cuda()
    z = _randn((B, L, ld), 23).cuda()
    g = z[..., :C]
    wg, wl = (torch.rand(64, generator=torch.Generator().manual_seed(s)).cuda() + 0.5 for s in (24, 25))
    y, out = (torch.full((B, L, C), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    rc = _lib.load().vig_locality_blend_linear_kept_fwd(o.data_ptr(), loc.data_ptr(), g.data_ptr(), wg.data_ptr(), wl.data_ptr(), w.data_ptr(),
                                                        y.data_ptr(), out.data_ptr(), B, H, L, 64, C, ld, 1e-5, 0, _lib.VIG_BF16,
                                                        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert torch.equal(out, ops.locality_blend_linear(o, loc, g, wg, wl, w, eps=1e-5))
    od, ld_, gd = o.double().cpu().permute(0, 2, 1, 3), loc.double().cpu().view(B, L, H, 64), torch.sigmoid(g.double().cpu()).view(B, L, H, 64)
    rms = lambda t, n: t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-5) * n.double().cpu()  # noqa: E731
    want = (rms(od, wg) * gd + rms(ld_, wl) * (1 - gd)).reshape(B, L, C)
    _check(y, want)
