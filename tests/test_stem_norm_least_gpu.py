"""The gradients of the patch embedding's norm on one row of one and two octets, where dx nearly cancels: against fp64 on the stored inputs."""
import pytest
import torch
import torch.nn.functional as F

from vig_amd import _ext

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("amp,last", [(True, False), (True, True), (False, False)])
@pytest.mark.parametrize("C", [8, 16])
def test_one_row(C, amp, last):
    announce(f"stem norm, one row of {C}, amp{amp} last{last}")
    g = torch.Generator().manual_seed(C)
    r = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    x = r(1, C, 1, 1).to(torch.bfloat16 if amp else torch.float32).contiguous(memory_format=torch.channels_last).requires_grad_()
    pre, w, b = (p.requires_grad_() for p in (r(C), r(C) + 1, r(C)))
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
        y = _ext.calls().stem_norm(x, pre, w, b, 1e-5, True, last)
    dy = r(1, C, 1, 1).to(y.dtype)
    got = [t.double().view(C) for t in torch.autograd.grad(y, (x, pre, w, b), dy)]

    t = [v.detach().double().view(C).requires_grad_() for v in (x, pre, w, b)]
    s = t[0] + t[1]
    z = F.silu(F.layer_norm(s, (C,), t[2], t[3], 1e-5))
    d = dy.double().view(C)
    want = torch.autograd.grad(z, t, d)
    # Some thirty fp32 roundings of terms no larger than these (xhat's of the row's largest value; SiLU's slope is below 1.1, its own below 0.5)
    rstd = 1 / (s.var(unbiased=False) + 1e-5).sqrt()
    xhat = (1 + rstd * s.abs().max()).detach()
    dw = (d * t[2]).abs().detach()
    e = 32 * 2.0 ** -24 * xhat * (1 + t[2].abs().max().detach())
    row = e * rstd.detach() * (dw + dw.mean() + xhat * (xhat * dw).mean())
    bounds = row + (2.0 ** -8 * want[0].abs() if amp else 0), row, e * xhat * d.abs(), e * d.abs()
    for name, a, v, bound in zip(("dx", "dpre", "dweight", "dbias"), got, want, bounds):
        assert ((a - v).abs() <= bound).all(), (name, ((a - v).abs() / bound).max().item())
