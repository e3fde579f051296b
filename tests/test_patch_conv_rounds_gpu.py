"""The stem's first convolution at the numbers of items where its workgroups stop having one each: 256 of more than four waves, 512 of up to four."""
import pytest
import torch
import torch.nn.functional as F

from vig_amd import ops

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Cout", [128, 160, 384])
@pytest.mark.parametrize("B", [255, 256, 257, 512, 513])
def test_items(B, Cout):
    announce(f"patch convolution, {B} items, Cout {Cout}")
    g = torch.Generator().manual_seed(B)
    x, w = torch.randn(B, 3, 7, 8, generator=g).bfloat16().cuda(), (torch.randn(Cout, 3, 9, 9, generator=g) * 0.1).bfloat16().cuda()
    got = ops.patch_conv(x, ops.pack_patch_conv_weight(w), (9, 9))
    want = F.conv2d(x.double(), w.double(), None, 8, 1).permute(0, 2, 3, 1)
    assert got.shape == want.shape == (B, 1, 1, Cout)
    assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()  # the stored value's rounding; fp32 sums of 243 terms
