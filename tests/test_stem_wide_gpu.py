"""The stem's first convolution at 384 output channels (twelve waves a workgroup) and, with it, the planned forward of a
768-wide model against its modules."""
import pytest
import torch

from vig_amd import layers, ops

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W,KW", [(1, 9, 8, 9), (3, 24, 248, 9), (2, 17, 264, 9), (1, 40, 64, 16), (40, 112, 112, 9)])
def test_patch_conv_384(B, H, W, KW):
    """Against fp64 on the stored inputs: one rounding of the output, and the fp32 sums of 243 products and more."""
    announce(f"patch_conv B{B} {H}x{W} KW{KW} Cout384")
    g = torch.Generator().manual_seed(11)
    x, w = torch.randn(B, 3, H, W, generator=g).bfloat16(), (torch.randn(384, 3, 9, KW, generator=g) * 0.1).bfloat16()
    assert ops.patch_conv_supported(x.cuda(), w.cuda(), 8, 1)
    got = ops.patch_conv(x.cuda(), ops.pack_patch_conv_weight(w.cuda()), (9, KW), 8, 1)
    want = torch.nn.functional.conv2d(x.double(), w.double(), None, 8, 1).permute(0, 2, 3, 1)
    assert tuple(got.shape) == tuple(want.shape)
    err = (got.double().cpu() - want).abs() / want.abs().clamp_min(1.0)
    assert err.max().item() <= 2.0 ** -8, err.max().item()


@pytest.mark.parametrize("B,side", [(1, 224), (3, 80)])
def test_planned_forward_768(B, side):
    announce(f"planned ViG-B forward B{B} {side}px")
    torch.manual_seed(5)
    with torch.device("cuda"):
        net = layers.ViG(img_size=side, embed_dim=768, num_heads=12, depth=2, num_classes=64, use_out_act=True,
                         use_act_in_conv=True).eval().to(torch.bfloat16)
        images = torch.randn(B, 3, side, side).bfloat16()
    planned = net(images)
    assert layers._PLANS.get(net) is not None
    with torch.no_grad():  # the modules one by one
        modules = net.head(net.forward_features(images))
    err = (planned.float() - modules.float()).norm() / modules.float().norm()
    assert err.item() <= 2e-2, err.item()  # bf16 activations of two blocks, products in another order


# one size for each tile shape of the rule, ragged rows and columns (64 x 192, 128 x 128, 128 x 192 in turn)
@pytest.mark.parametrize("B,H,W,Cin,Cout", [(33, 28, 27, 64, 760), (47, 28, 28, 64, 760), (63, 27, 28, 64, 760)])
def test_conv3x3s2_tiles(B, H, W, Cin, Cout):
    announce(f"3x3 stride-2 convolution B{B} {H}x{W} {Cin}->{Cout}")
    g = torch.Generator().manual_seed(12)
    x, w = torch.randn(B, Cin, H, W, generator=g).bfloat16(), (torch.randn(Cout, Cin, 3, 3, generator=g) * (9 * Cin) ** -0.5).bfloat16()
    got = ops.conv3x3s2(x.cuda().contiguous(memory_format=torch.channels_last), w.cuda().contiguous(memory_format=torch.channels_last))
    want = torch.nn.functional.conv2d(x.double(), w.double(), None, 2, 1)
    err = (got.double().cpu() - want).abs() / want.abs().clamp_min(1.0)
    assert err.max().item() <= 2.0 ** -7, err.max().item()
