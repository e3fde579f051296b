"""Elementwise kernels that deal channel octets of token rows out to workgroups (split and merge of heads, directional gates, locality
blend, forward and backward) where that can go wrong: images of a token or two inside one workgroup, ragged ends, odd widths, rows of
more octets than threads, four octets a thread, and the smallest workspace."""
import pytest
import torch
import torch.nn.functional as F

import vig_amd
from oracle import gla_oracle as O
from vig_amd import _lib

from .util import announce, f64, max_abs

pytestmark = pytest.mark.gpu

# (batch, heads, tokens): a workgroup holds many images | ragged | odd heads | wider than 256 octets | four octets a thread, ragged
SHAPES = [(70, 3, 1), (33, 2, 7), (1, 5, 301), (3, 40, 33), (3, 12, 3701)]


def _randn(shape, seed, dtype):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,H,L", SHAPES)
@pytest.mark.parametrize("Dk,Dv", [(32, 64), (16, 32)])
def test_heads(B, H, L, Dk, Dv, dtype):
    announce(f"split and merge of heads B{B} H{H} L{L} Dk{Dk} {dtype}")
    row, wide = H * (2 * Dk + Dv), H * (2 * Dk + Dv) + 24
    z = _randn((B, L, wide), 1, dtype)
    q, k, v = (torch.empty(B, H, L, d, dtype=dtype, device="cuda") for d in (Dk, Dk, Dv))
    lib, code = _lib.load(), int(dtype == torch.bfloat16)
    assert lib.vig_split_heads_fwd(z.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), B, L, H, Dk, Dv, wide, code, _stream()) == 0
    at = 0
    for t, D in ((q, Dk), (k, Dk), (v, Dv)):
        assert torch.equal(t, z[..., at:at + H * D].reshape(B, L, H, D).transpose(1, 2))
        at += H * D
    back = torch.full_like(z, 3.0)
    assert lib.vig_split_heads_bwd_strided(q.data_ptr(), k.data_ptr(), v.data_ptr(), back.data_ptr(), wide, B, L, H, Dk, Dv, code,
                                           _stream()) == 0
    assert torch.equal(back[..., :row], z[..., :row]) and (back[..., row:] == 3.0).all()


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.bfloat16, 4e-3)])  # (bf16: half a unit in the last place below 1)
@pytest.mark.parametrize("B,H,L", SHAPES)
def test_gates(B, H, L, dtype, tol):
    announce(f"directional gates B{B} H{H} L{L} {dtype}")
    Dk, code, lib = 32, int(dtype == torch.bfloat16), _lib.load()
    x, d = _randn((B, L, 2 * H * Dk), 2, dtype), _randn((2, B, H, L, Dk), 3, dtype)
    out, dx = torch.empty_like(d), torch.empty_like(x)
    args = (B, L, H, Dk, 1 / 16, -0.1, code, code, _stream())
    assert lib.vig_dirgate_fwd(x.data_ptr(), out.data_ptr(), *args) == 0
    assert lib.vig_dirgate_bwd(x.data_ptr(), d.data_ptr(), dx.data_ptr(), *args) == 0
    heads = x.double().view(B, L, 2, H, Dk).permute(2, 0, 3, 1, 4)
    plain = F.logsigmoid(heads) / 16
    assert (out.double() - plain.clamp_min(-0.1)).abs().max() <= tol
    want = torch.where(plain < -0.1, 0.0, d.double() / 16 * torch.sigmoid(-heads))
    near = (plain + 0.1).abs() < 1e-6  # (either side of the clamp)
    got = dx.double().view(B, L, 2, H, Dk).permute(2, 0, 3, 1, 4)
    assert (got - want)[~near].abs().max() <= tol


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5), (torch.bfloat16, 3e-2)])
@pytest.mark.parametrize("B,H,L", SHAPES)
@pytest.mark.parametrize("Dv", [32, 64])
def test_blend(B, H, L, Dv, dtype, tol):
    announce(f"locality blend B{B} H{H} L{L} Dv{Dv} {dtype}")
    o, loc, gl = _randn((B, H, L, Dv), 4, dtype), _randn((B, L, H * Dv), 5, dtype), _randn((B, L, H * Dv), 6, dtype)
    wg, wl = (_randn((Dv,), s, torch.float32) * 0.1 + 1 for s in (7, 8))
    got = vig_amd.locality_blend(o, loc, gl, wg, wl, 1e-6, True)
    want = O.locality_blend_reference(*(f64(t) for t in (o, loc, gl, wg, wl)), 1e-6, True)
    assert max_abs(f64(got), want) <= tol


@pytest.mark.parametrize("least", [False, True])
@pytest.mark.parametrize("dtype,eps", [(torch.float32, 2.0 ** -21), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("B,H,L", SHAPES)
def test_blend_gradients(B, H, L, dtype, eps, least):
    announce(f"locality blend gradients B{B} H{H} L{L} {dtype} least workspace {least}")
    Dv, code, lib = 64, int(dtype == torch.bfloat16), _lib.load()
    o, loc, gl, dy = (_randn(s, n, dtype) for n, s in enumerate([(B, H, L, Dv)] + [(B, L, H * Dv)] * 3))
    wg, wl = (_randn((Dv,), s, torch.float32) * 0.1 + 1 for s in (7, 8))
    do, dl, dg = torch.empty_like(o), torch.empty_like(loc), torch.empty_like(gl)
    dw = torch.empty(2, Dv, device="cuda")
    size = B * ((L + 31) // 32) * 2 * Dv * 4 if least else lib.vig_locality_blend_bwd_workspace(B, L, Dv)
    guard = torch.full((size + 1024,), 77, dtype=torch.uint8, device="cuda")
    rc = lib.vig_locality_blend_bwd_strided(o.data_ptr(), loc.data_ptr(), gl.data_ptr(), wg.data_ptr(), wl.data_ptr(), dy.data_ptr(),
                                            do.data_ptr(), dl.data_ptr(), dg.data_ptr(), dw.data_ptr(), guard.data_ptr(), size, B, H, L,
                                            Dv, 0, 0, 1e-6, 1, code, _stream())
    assert rc == 0 and (guard[size:] == 77).all()
    t = [x.double().requires_grad_() for x in (o, loc, gl, wg, wl)]

    def rms(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-6) * w

    s = torch.sigmoid(t[2]).view(B, L, H, Dv)
    y = (rms(t[0].transpose(1, 2), t[3]) * s + rms(t[1].view(B, L, H, Dv), t[4]) * (1 - s)).reshape(B, L, H * Dv)
    F.silu(y).backward(dy.double())
    for got, want in zip((do, dl, dg), t):  # a rounding to the storage type and a few of fp32, of values up to the largest
        assert ((got.double() - want.grad).abs() <= eps * want.grad.abs().max()).all()
    for got, want in zip(dw, t[3:]):  # sums of B * L * H terms, none of them above the largest of 5 sigma
        assert (got.double() - want.grad).abs().max() <= 2.0 ** -20 * 5 * (B * L * H) ** 0.5 + 2.0 ** -20 * want.grad.abs().max()


def test_blend_gradients_refuse_less_room():
    x = torch.zeros(2, 3, 40, 64, device="cuda")
    w, dw = torch.ones(64, device="cuda"), torch.empty(2, 64, device="cuda")
    size = 2 * 2 * 2 * 64 * 4 - 4
    assert _lib.load().vig_locality_blend_bwd_strided(*([x.data_ptr()] * 3), w.data_ptr(), w.data_ptr(), *([x.data_ptr()] * 4), dw.data_ptr(),
                                                      x.data_ptr(), size, 2, 3, 40, 64, 0, 0, 1e-6, 0, 0, _stream()) == _lib.VIG_ENOSPC
