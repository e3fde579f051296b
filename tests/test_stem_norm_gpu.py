"""The layer norms of the patch embedding in training (bias in front, SiLU behind, one node): values and gradients against fp64 on the stored inputs at every
lane layout, the calls that stay with the modules, and a graph of the gradients."""
import pytest
import torch
import torch.nn.functional as F

from vig_amd import _ext, layers

from .util import announce

pytestmark = pytest.mark.gpu


def _reference(x, pre, w, b, silu, dy):
    t = [v.double().requires_grad_() if v is not None else None for v in (x, pre, w, b)]
    s = t[0].permute(0, 2, 3, 1) if t[1] is None else t[0].permute(0, 2, 3, 1) + t[1]
    z = F.layer_norm(s, (x.shape[1],), t[2], t[3], 1e-5)
    z = (F.silu(z) if silu else z).permute(0, 3, 1, 2)
    return [z.detach()] + list(torch.autograd.grad(z, [v for v in t if v is not None], dy.double()))


@pytest.mark.parametrize("amp,last", [(True, False), (True, True), (False, False)])
@pytest.mark.parametrize("B,C,h,w,bias,silu", [(1, 8, 1, 1, True, True), (2, 96, 5, 7, True, True), (3, 192, 28, 28, True, True), (2, 256, 3, 3, False, False),
                                               (5, 384, 14, 13, True, False), (1, 768, 9, 4, True, True), (60, 1024, 14, 14, False, True)])
def test_against_fp64(B, C, h, w, bias, silu, amp, last):
    announce(f"stem norm B{B} C{C} {h}x{w} bias{bias} silu{silu} amp{amp} last{last}")
    g = torch.Generator().manual_seed(C)
    r = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    x = r(B, C, h, w).to(torch.bfloat16 if amp else torch.float32).contiguous(memory_format=torch.channels_last).requires_grad_()
    params = [p.requires_grad_() if p is not None else None for p in (r(C) if bias else None, r(C) + 1, r(C))]
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
        y = _ext.calls().stem_norm(x, *params, 1e-5, silu, last)
    out = torch.bfloat16 if amp and not last else torch.float32
    assert y.dtype == out and y.shape == x.shape and y.is_contiguous(memory_format=torch.channels_last)
    dy = r(B, C, h, w).to(out)  # (not in channels-last memory)
    got = [y.detach()] + list(torch.autograd.grad(y, [t for t in (x, *params) if t is not None], dy))
    for i, (a, b) in enumerate(zip(got, _reference(x.detach(), *(None if p is None else p.detach() for p in params), silu, dy))):
        # a stored bf16 value: its rounding; fp32 sums of up to rows * C terms and the transcendentals' last bits
        bound = 2.0 ** -8 if a.dtype == torch.bfloat16 else 2e-5
        if C * h * w > 8 or i == 0:
            assert (a.double() - b).norm() <= bound * b.norm() + 1e-12, (i, ((a.double() - b).norm() / b.norm()).item())


def test_stays_with_the_modules():
    announce("stem norm: calls the node does not take, hooks, and the same result as the modules")
    torch.manual_seed(0)
    stem, x = layers.V2PatchEmbed(embed_dim=192).cuda().train(), torch.randn(2, 3, 64, 48, device="cuda")
    seen = []

    def run(fn):
        for p in stem.parameters():
            p.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = fn(x)
        y.float().square().sum().backward()
        return [y.detach().float()] + [p.grad for p in stem.parameters()]

    want = run(stem.proj)
    for a, b in zip(run(stem._recorded), want):
        assert (a - b).norm() <= 2e-2 * b.norm()  # two convolutions' bf16 roundings
    handle = stem.proj[1].register_forward_hook(lambda *a: seen.append(1))
    assert all(torch.equal(a, b) for a, b in zip(run(stem._recorded), run(stem.proj))) and len(seen) == 2
    handle.remove()
    calls, n = _ext.calls(), stem.proj[1]
    m = torch.randn(2, 96, 4, 4, device="cuda")
    take = lambda m: calls.stem_norm(m, None, n.weight, n.bias, 1e-5, True, False)  # noqa: E731
    assert take(m) is None  # not channels-last
    m = m.contiguous(memory_format=torch.channels_last)
    assert take(m) is not None and take(m.bfloat16()) is None and take(m[:, :90]) is None and take(m.double()) is None
    with torch.autocast("cuda", dtype=torch.float16):
        assert take(m) is None


def test_graph_of_the_gradients():
    announce("stem norm: second derivatives")
    g = torch.Generator().manual_seed(1)
    x = torch.randn(2, 16, 3, 3, generator=g).cuda().contiguous(memory_format=torch.channels_last).requires_grad_()
    p = [torch.randn(16, generator=g).cuda().requires_grad_() for _ in range(3)]
    d = torch.randn(2, 16, 3, 3, generator=g).cuda()

    def second(y):
        first = torch.autograd.grad(y, [x, *p], d, create_graph=True)
        return torch.autograd.grad(sum(t.square().sum() for t in first), [x, *p])

    z = F.silu(F.layer_norm(x.permute(0, 2, 3, 1) + p[0], (16,), p[1], p[2], 1e-5)).permute(0, 3, 1, 2)
    for a, b in zip(second(_ext.calls().stem_norm(x, *p, 1e-5, True, False)), second(z)):
        assert torch.allclose(a, b, rtol=1e-3, atol=1e-4)
