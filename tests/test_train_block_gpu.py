"""The recorded block as two autograd nodes and the kernels it adds, at the sizes where they can go wrong: against the same
block run module by module in fp32, and against float64 sums."""
import pytest
import torch
from torch.nn.utils import prune

from vig_amd import _lib, layers

from .util import announce

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).norm() / b.norm().clamp_min(1e-30))


def _ptr(t):
    return t.data_ptr() if t is not None else None


# (batch, grid, width, heads, Dk, SiLU in conv and on output, conv bias, clamp): two tokens, ragged token tiles, a grid of several
# bands, widths that leave padding columns or none, every head width
BLOCKS = [
    (1, (1, 2), 64, 1, 32, False, False, None),
    (3, (7, 5), 192, 3, 32, True, True, None),
    (2, (14, 14), 96, 3, 16, True, False, -0.3),
    (2, (33, 9), 128, 2, 64, False, True, None),
    (1, (4, 61), 320, 5, 32, False, False, None),
]


@pytest.mark.parametrize("mode,tol", [("fp32", 2e-5), ("bf16", 3e-2), ("amp", 2e-2)])
@pytest.mark.parametrize("B,hw,C,H,Dk,act,bias,clamp", BLOCKS)
def test_recorded_block(B, hw, C, H, Dk, act, bias, clamp, mode, tol):
    announce(f"recorded block B{B} {hw} C{C} H{H} Dk{Dk} act={act} bias={bias} clamp={clamp} {mode}")
    torch.manual_seed(C + hw[0])
    blk = layers.GLABlock(C, H, Dk * H / C, 1.0, use_out_act=act, use_act_in_conv=act, use_bias_in_dwconv=bias,
                          intermediate_size=2 * C)
    blk.attn.clamp_min = clamp
    with torch.no_grad():
        for p in blk.parameters():
            p.copy_(torch.randn_like(p) * (0.3 if p.dim() == 1 else p.shape[-1] ** -0.5 if p.dim() == 2 else 0.3))
        for m in (blk.attn_norm, blk.mlp_norm, blk.attn.g_norm, blk.attn.l_norm):
            m.weight.add_(1.0)
    x, res, cot, cot2 = (torch.randn(B, hw[0] * hw[1], C) for _ in range(4))
    wide = torch.bfloat16 if mode == "bf16" else torch.float32  # the residual stream's type
    narrow = torch.float32 if mode == "fp32" else torch.bfloat16

    def run(fused, residual, param, x_type, stream):
        m = blk.to("cuda", param).train()
        m.__dict__.pop("_recorded", None)
        if not fused:
            m._recorded = lambda *a, **k: None
        m.zero_grad()
        xs = [x.cuda().to(x_type if residual else stream).requires_grad_()]
        if residual:
            xs.append(res.cuda().to(stream).requires_grad_())
        with torch.autocast("cuda", torch.bfloat16, enabled=mode == "amp" and fused):
            y, total = m.forward_carry(xs[0], xs[1] if residual else None, patch_resolution=hw)
        ((y.float() * cot.cuda()).sum() + (total.float() * cot2.cuda()).sum()).backward()
        out = {"y": y, "total": total, **{f"x{i}": t.grad for i, t in enumerate(xs)}}
        out.update({n: p.grad for n, p in m.named_parameters()})
        return out, y.grad_fn.name()

    with torch.no_grad():
        for p in blk.parameters():
            p.copy_(p.to(torch.bfloat16 if mode == "bf16" else torch.float32))
    x, res = x.to(narrow).float(), res.to(wide).float()
    for residual in (False, True):
        want, _ = run(False, residual, torch.float32, torch.float32, torch.float32)
        got, node = run(True, residual, torch.bfloat16 if mode == "bf16" else torch.float32, narrow, wide)
        assert "Mlp" in node, node  # the nodes ran, not the modules
        for n, w in want.items():
            e = _rel(got[n].detach(), w.detach())
            assert e <= tol * (1 if n in ("y", "total") or mode == "fp32" else 2), (residual, n, e)


class _Doubled(layers.RMSNorm):
    def forward(self, *args, **kwargs):
        y = super().forward(*args, **kwargs)
        return (2 * y[0], *y[1:]) if isinstance(y, tuple) else 2 * y


@pytest.mark.parametrize("change", ["adapter", "norm", "gate layers", "pruned", "hook on all modules", "mixer"])
def test_block_runs_module_by_module_where_something_hangs_on_a_call(change):
    announce(f"recorded block with a changed module: {change}")
    torch.manual_seed(3)
    blk = layers.GLABlock(192, 3, 0.5, 1.0, intermediate_size=512).cuda().train()
    with torch.no_grad():  # (as initialised, the mixer hardly shows in the output)
        for p in blk.parameters():
            p.add_(torch.randn_like(p) * p.shape[-1] ** -0.5)
    at, seen, handle = blk.attn, [], None
    x = torch.randn(2, 30, 192, device="cuda")

    def run():
        blk.zero_grad()
        y, _ = blk.forward_carry(x, None, patch_resolution=(5, 6))
        y.square().sum().backward()
        return y, [p.grad.clone() for p in blk.parameters() if p.grad is not None]

    before, _ = run()
    assert "Mlp" in before.grad_fn.name()
    if change == "adapter":
        at.qkv_proj.forward = lambda h, lin=at.qkv_proj: torch.nn.Linear.forward(lin, h) + 0.5 * h.repeat(1, 1, 2)
    elif change == "norm":
        norm = _Doubled(192).cuda()
        norm.load_state_dict(blk.mlp_norm.state_dict())
        blk.mlp_norm = norm
    elif change == "gate layers":
        at.gk_proj.append(torch.nn.Hardtanh(-0.01, 0.01))
    elif change == "pruned":
        torch.manual_seed(4)
        prune.random_unstructured(blk.mlp.down_proj, "weight", 0.5)
    elif change == "mixer":
        at._mix_autograd = lambda h, hw, s: 2 * type(at)._mix_autograd(at, h, hw, s)
    else:
        handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: seen.append(1))
    try:
        got, grads = run()
        blk._recorded = lambda *a, **k: None
        want, wanted = run()
    finally:
        if handle is not None:
            handle.remove()
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(grads, wanted, strict=True))
    assert seen if change == "hook on all modules" else not torch.allclose(got, before, rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("rows,N,K", [(1, 8, 8), (33, 40, 16), (65, 136, 264), (1000, 384, 16), (2500, 1168, 384), (4097, 200, 192)])
def test_linear_bwd_weight(rows, N, K):
    announce(f"linear weight and bias gradients rows={rows} N={N} K={K}")
    g = torch.Generator().manual_seed(rows)
    dy = torch.randn(rows, N + 24, generator=g).bfloat16().cuda()[:, 8:8 + N]
    x = torch.randn(rows, K + 8, generator=g).bfloat16().cuda()[:, :K]
    lib = _lib.load()
    dw = torch.empty(N, K, device="cuda")
    db = torch.empty(N, device="cuda")
    need = lib.vig_linear_bwd_weight_workspace(rows, N, K)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    _lib.check(lib.vig_linear_bwd_weight(dy.data_ptr(), dy.stride(0), x.data_ptr(), x.stride(0), dw.data_ptr(), db.data_ptr(),
                                         ws.data_ptr(), need, rows, N, K, torch.cuda.current_stream().cuda_stream), "wgrad")
    d64, x64 = dy.double().cpu(), x.double().cpu()
    assert _rel(dw, d64.t() @ x64) <= 2e-6
    assert _rel(db, d64.sum(0)) <= 2e-6


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.bfloat16, 6e-3)])
@pytest.mark.parametrize("B,h,w,C", [(1, 1, 1, 8), (2, 3, 7, 72), (2, 40, 17, 64), (1, 9, 126, 136), (1, 5, 130, 64)])
def test_dwconv_backward(B, h, w, C, dtype, tol):
    announce(f"depthwise convolution's gradients B{B} {h}x{w} C{C} {dtype}")
    g = torch.Generator().manual_seed(h * w)
    x, dy, pre = (torch.randn(B, h * w, C, generator=g).to(dtype) for _ in range(3))
    wt = torch.randn(C, 9, generator=g)
    lib = _lib.load()
    for use_pre in (False, True):
        z = pre.double().requires_grad_()
        torch.nn.functional.silu(z).backward(dy.double())
        d = (z.grad.to(dtype) if use_pre else dy).double()
        img = lambda t: t.reshape(B, h, w, C).permute(0, 3, 1, 2)  # noqa: E731
        x64, w64 = img(x.double()).clone().requires_grad_(), wt.double().reshape(C, 1, 3, 3).requires_grad_()
        torch.nn.functional.conv2d(x64, w64, padding=1, groups=C).backward(img(d))
        xc, dc, pc, wc = x.cuda(), dy.cuda(), pre.cuda(), wt.cuda()
        dx, both = torch.empty_like(xc), torch.empty(C * 10, device="cuda")
        need = lib.vig_dwconv3x3_bwd_weight_workspace(B, C)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        _lib.check(lib.vig_dwconv3x3_bwd(xc.data_ptr(), dc.data_ptr(), _ptr(pc if use_pre else None), wc.data_ptr(), dx.data_ptr(),
                                         both.data_ptr(), ws.data_ptr(), need, B, h, w, C, 0 if dtype == torch.float32 else 1,
                                         torch.cuda.current_stream().cuda_stream), "vig_dwconv3x3_bwd")
        assert _rel(dx, x64.grad.permute(0, 2, 3, 1).reshape(B, h * w, C)) <= tol
        assert _rel(both[:C * 9], w64.grad.reshape(-1)) <= tol
        assert _rel(both[C * 9:], d.sum((0, 1))) <= tol
