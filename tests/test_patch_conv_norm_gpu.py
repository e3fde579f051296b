"""The stem's first convolution with the layer norm and SiLU behind it in one kernel against the two kernels: every width of channels, one and several
items a workgroup, rows cut into pieces, without a bias or an activation."""
import pytest
import torch

from vig_amd import _lib, ops

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W,Cout,full", [(1, 9, 8, 64, True), (2, 33, 248, 96, False), (30, 224, 224, 128, True), (1, 24, 264, 160, True),
                                             (25, 200, 224, 192, True), (3, 17, 512, 224, False), (1, 40, 64, 256, True)])
def test_against_two_kernels(B, H, W, Cout, full):
    announce(f"patch convolution and norm B{B} {H}x{W} Cout{Cout}")
    g = torch.Generator().manual_seed(Cout)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x, w = r(B, 3, H, W).bfloat16().cuda(), ops.pack_patch_conv_weight((r(Cout, 3, 9, 9) * 0.1).bfloat16().cuda())
    nw, nb, pre = (r(Cout).cuda() for _ in range(3))
    p, lib, st = (lambda t: t.data_ptr()), _lib.load(), torch.cuda.current_stream().cuda_stream
    rows = B * ((H + 2 - 9) // 8 + 1) * ((W + 2 - 9) // 8 + 1)
    got, conv, want = (torch.full((rows, Cout), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(3))
    shape, pre = (B, 3, H, W, 9, 9, 8, 1, Cout), p(pre) if full else None
    assert lib.vig_patch_conv_norm_fwd(p(x), p(w), p(nw), p(nb), pre, p(got), *shape, 1e-6, full, st) == _lib.VIG_OK
    assert lib.vig_patch_conv_fwd(p(x), p(w), p(conv), *shape, 1, st) == _lib.VIG_OK
    assert lib.vig_layernorm_fwd(p(conv), p(nw), p(nb), p(want), rows, Cout, 1e-6, full, pre, None, 0, 1, st) == _lib.VIG_OK
    assert torch.equal(got, want)  # the same sums in the same order


def test_refused():
    x, f, lib = torch.zeros(384 * 64 * 27 * 16, dtype=torch.bfloat16, device="cuda"), torch.zeros(384, device="cuda"), _lib.load()
    p, q, st = x.data_ptr(), f.data_ptr(), torch.cuda.current_stream().cuda_stream
    call = lambda n, W=64, b=q: lib.vig_patch_conv_norm_fwd(p, p, q, b, None, p, 1, 3, 40, W, 9, 9, 8, 1, n, 1e-6, 1, st)  # noqa: E731
    assert call(384) == _lib.VIG_ENOTSUP and call(80) == _lib.VIG_ENOTSUP and call(64, W=68) == _lib.VIG_ENOTSUP
    assert call(64, b=None) == _lib.VIG_EINVAL
