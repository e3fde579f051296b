"""The row kernels spread over more workgroups when there are few images, where they can go wrong: against float64 sums of the
same bf16 values."""
import pytest
import torch

from vig_amd import ops

from .util import announce

pytestmark = pytest.mark.gpu


def _randn(shape, seed, scale=1.0):
    return (torch.randn(shape, generator=torch.Generator().manual_seed(seed)) * scale).bfloat16()


def _check(got, want64, ulps=1.0):
    """Within `ulps` bf16 roundings (2^-8 relative) and the fp32 sums' error, 1e-5 of the result's scale."""
    got = got.double().cpu()
    assert ((got - want64).abs() <= ulps * 2.0 ** -8 * want64.abs() + 1e-5 * want64.abs().max()).all()


# the depthwise convolution in bands of one to a few rows, one workgroup for each up to 128
@pytest.mark.parametrize("B,h,w,C", [(1, 14, 14, 192), (1, 1, 5, 64), (5, 13, 7, 384), (43, 9, 6, 192), (1, 64, 64, 72)])
def test_few_bands(B, h, w, C):
    announce(f"dwconv3x3 B{B} {h}x{w} C{C}")
    x, wt = _randn((B, h * w, C), 6), torch.randn(C, 1, 3, 3, generator=torch.Generator().manual_seed(7)) / 3
    got = ops.dwconv3x3(x.cuda(), wt[:, 0].cuda(), (h, w))
    want = torch.nn.functional.conv2d(x.double().view(B, h, w, C).permute(0, 3, 1, 2), wt.double(), None, 1, 1, 1, C)
    _check(got, want.permute(0, 2, 3, 1).reshape(B, h * w, C))


# gate preparation with the channel tiles of a token group over several workgroups: one round, an uneven last one, all alone
@pytest.mark.parametrize("B,L,H,Dk", [(1, 5, 3, 32), (1, 196, 5, 48), (2, 33, 12, 64), (600, 64, 6, 32)])
def test_gate_rounds(B, L, H, Dk):
    announce(f"dirgate_lowrank B{B} L{L} H{H} Dk{Dk}")
    low, w, b = _randn((B, L, ops.GATE_RANK), 8), _randn((2 * H * Dk, ops.GATE_RANK), 9, 0.25), _randn((2 * H * Dk,), 10)
    out = ops.dirgate_lowrank(low.cuda(), w.cuda(), b.cuda(), H)
    x = torch.nn.functional.linear(low.double(), w.double(), b.double())
    want = torch.nn.functional.logsigmoid(x.float().bfloat16().double()) / 16
    want = want.view(B, L, 2, H, Dk).permute(2, 0, 3, 1, 4)
    got = out.double().cpu()
    # a bf16 rounding of the result and, where the sum rounds the other way, one of the pre-activation (below 8, slope <= 1/16)
    assert ((got - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -8 * 8 / 16).all()
