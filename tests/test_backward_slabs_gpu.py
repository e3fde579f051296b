"""The matrix-core backward's workgroups of two, three (64 key channels only), four, seven and eight tiles at the edges of their
ranges, and with more slabs than workgroups (each walks several)."""
import pytest
import torch

import vig_amd
from oracle import gla_oracle as O
from vig_amd.synthetic import make_gla_inputs

from .test_backward_gpu import _check_mfma, _do
from .util import announce, f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("both", [True, False])
@pytest.mark.parametrize("B,H,L,Dk", [(2, 2, 63, 32), (2, 2, 65, 64), (1, 3, 65, 32), (1, 2, 127, 64), (1, 3, 128, 32), (1, 2, 129, 64),
                                      (1, 2, 129, 32)])
def test_lengths(B, H, L, Dk, both):
    announce(f"backward slabs B{B} H{H} L{L} Dk{Dk} both={both}")
    q, k, v, gf, gb = make_gla_inputs(B, H, L, Dk, 64, seed=40 + L, dtype=torch.bfloat16)
    do = _do(v.shape, 3, torch.bfloat16)
    if both:
        want = O.bidir_gla_backward(f64(q), f64(k), f64(v), f64(gf), f64(gb), f64(do), out_scale=0.5)
    else:
        want = O.gla_recurrent_backward(f64(q), f64(k), f64(v), f64(gf), f64(do))
    got = vig_amd.gla_bidir_backward(q.cuda(), k.cuda(), v.cuda(), gf.cuda(), gb.cuda() if both else None, do.cuda(),
                                     out_scale=0.5 if both else 1.0)
    _check_mfma(got if both else got[:4], want, q)


@pytest.mark.parametrize("B,H,L,Dk", [(360, 3, 57, 32), (180, 6, 40, 64), (90, 6, 100, 64)])
def test_more_slabs_than_workgroups(B, H, L, Dk):
    """Every ninth slab beyond the quadratic form's range: those from the recurrent kernel bit for bit, the rest within the bound."""
    announce(f"backward slabs, {B * H} of {L} tokens, Dk{Dk}")
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, L, Dk, 64, seed=5, dtype=torch.bfloat16))
    strong = (torch.arange(B * H, device="cuda") % 9 == 4).reshape(B, H)
    gf = torch.where(strong[:, :, None, None], torch.full_like(gf, -4.0), gf)
    do = _do(v.shape, 4, torch.bfloat16).cuda()
    exact = vig_amd.gla_bidir_backward(q, k, v, gf, gb, do, out_scale=0.5, exact=True)
    got = vig_amd.gla_bidir_backward(q, k, v, gf, gb, do, out_scale=0.5)
    for g, e in zip(got, exact):
        assert torch.equal(g[strong], e[strong])
    keep = ~strong
    _check_mfma([g[keep] for g in got], [f64(e[keep]) for e in exact], q[keep].cpu())


@pytest.mark.parametrize("B,H,L,Dk,both", [(1, 2, 6200, 32, True), (1, 1, 12400, 64, True), (1, 1, 6200, 32, False), (2, 3, 513, 32, True),
                                           (1, 3, 385, 32, True), (1, 2, 640, 32, False), (1, 2, 385, 64, True)])
def test_segments(B, H, L, Dk, both):
    """Long sequences at the edges of their segmentations: more segments than one chunk of the scan holds, last segments of one
    token and of whole tiles."""
    announce(f"backward segments B{B} H{H} L{L} Dk{Dk} both={both}")
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, L, Dk, 64, seed=90, dtype=torch.bfloat16))
    do = _do(v.shape, 6, torch.bfloat16).cuda()
    gb, out = (gb, 0.5) if both else (None, 1.0)
    want = vig_amd.gla_bidir_backward(q, k, v, gf, gb, do, out_scale=out, exact=True)
    got = vig_amd.gla_bidir_backward(q, k, v, gf, gb, do, out_scale=out)
    n = 5 if both else 4
    _check_mfma(got[:n], [f64(t) for t in want[:n]], q.cpu())


@pytest.mark.parametrize("both", [True, False])
@pytest.mark.parametrize("B,H,L,Dk", [(1, 2, 160, 64), (1, 2, 193, 32), (1, 2, 224, 64), (1, 2, 224, 32), (1, 2, 225, 64), (1, 3, 255, 32)])
def test_seven_and_eight_tiles(B, H, L, Dk, both):
    test_lengths(B, H, L, Dk, both)


@pytest.mark.parametrize("both", [True, False])
@pytest.mark.parametrize("B,H,L", [(1, 2, 65), (1, 1, 80), (2, 3, 96), (1, 2, 97), (90, 6, 95)])
def test_three_tiles(B, H, L, both):
    test_lengths(B, H, L, 64, both)


@pytest.mark.parametrize("both", [True, False])
@pytest.mark.parametrize("B,H,L", [(1, 1, 1), (1, 2, 32), (1, 1, 33), (2, 3, 64), (180, 6, 49)])
def test_two_tiles(B, H, L, both):
    """64 key channels: of the first direction's dq three units of four wait in LDS, one in the output tensor."""
    test_lengths(B, H, L, 64, both)


@pytest.mark.parametrize("B,H,L,Dk", [(90, 6, 70, 64), (87, 6, 197, 64), (87, 6, 197, 32), (90, 3, 230, 64), (90, 3, 230, 32)])
def test_slabs_given_up_in_either_direction(B, H, L, Dk):
    """Several slabs a workgroup, some beyond the range in their first direction, some in their second (whose loads are then
    on their way already), some in both: those from the recurrent kernel bit for bit, the rest within the bound."""
    announce(f"backward slabs, {B * H} of {L} tokens, Dk{Dk}, strong in either direction")
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, L, Dk, 64, seed=8, dtype=torch.bfloat16))
    slab = torch.arange(B * H, device="cuda").reshape(B, H)
    first, second = slab % 7 == 2, slab % 5 == 1
    gf = torch.where(first[:, :, None, None], torch.full_like(gf, -4.0), gf)
    gb = torch.where(second[:, :, None, None], torch.full_like(gb, -4.0), gb)
    do = _do(v.shape, 4, torch.bfloat16).cuda()
    exact = vig_amd.gla_bidir_backward(q, k, v, gf, gb, do, out_scale=0.5, exact=True)
    got = vig_amd.gla_bidir_backward(q, k, v, gf, gb, do, out_scale=0.5)
    strong = first | second
    for g, e in zip(got, exact):
        assert torch.equal(g[strong], e[strong])
    _check_mfma([g[~strong] for g in got], [f64(e[~strong]) for e in exact], q[~strong].cpu())


def test_two_tile_slabs_given_up_in_either_direction():
    test_slabs_given_up_in_either_direction(360, 3, 60, 64)
