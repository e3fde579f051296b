"""The fp32 matrix product (three bf16 pieces, six products) against fp64, in its three operand orders: edges of tiles, stages and
splits, operands inside wider matrices, bias, addend, column sums, infinities and overflow; what it refuses."""
import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _wide(rows, cols, pad, gen):
    return torch.randn(rows, cols + pad, generator=gen).cuda()[:, :cols]


def _matmul(a, ta, b, tb, bias=None, add=None, sums=False, out=None):
    M, K, N = a.shape[int(ta)], a.shape[1 - int(ta)], b.shape[int(tb)]
    lib = _lib.load()
    out = torch.full((M, N + 5), 7.0, device="cuda") if out is None else out
    s = torch.empty(M, device="cuda") if sums else None
    need = lib.vig_matmul_f32_workspace(M, N, K)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    p = lambda t: None if t is None else t.data_ptr()  # noqa: E731
    rc = lib.vig_matmul_f32(p(a), a.stride(0), ta, p(b), b.stride(0), tb, p(bias), p(add), 0 if add is None else add.stride(0), p(out),
                            out.stride(0), p(s), M, N, K, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return rc, out, s


@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (63, 65, 24), (64, 64, 32), (65, 132, 40), (400, 48, 512), (129, 16, 2056), (1000, 384, 16)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 1)])
def test_against_fp64(M, N, K, ta, tb):
    announce(f"fp32 product {M} {N} {K} across {ta} {tb}")
    gen = torch.Generator().manual_seed(M + N + K)
    a = _wide(K, M, 3, gen) if ta else _wide(M, K, 4, gen)
    b = _wide(K, N, 5, gen) if tb else _wide(N, K, 8, gen)
    A, Bt = (a.t() if ta else a).double(), (b if tb else b.t()).double()
    bias, add = torch.randn(N, generator=gen).cuda(), _wide(M, N, 1, gen)
    # a rounding of the leading accumulator for every 16 contraction steps and for every part of a split (at most 32), bias, addend
    # and the small accumulator, each within EPS of the sum of magnitudes; what the pieces leave out is below one of these
    bound = (K / 16 + 32 + 4) * EPS * (A.abs() @ Bt.abs() + bias.abs() + add.abs())
    rc, out, s = _matmul(a, ta, b, tb, bias, add, sums=bool(ta))
    assert rc == 0 and (out[:, N:] == 7.0).all()
    assert ((out[:, :N].double() - (A @ Bt + bias + add)).abs() <= bound).all()
    if ta:
        assert ((s.double() - A.sum(1)).abs() <= K * EPS * A.abs().sum(1)).all()
    rc, again, _ = _matmul(a, ta, b, tb, bias, add, sums=bool(ta))
    assert rc == 0 and torch.equal(out, again)
    if not ta:  # the addend is the output
        own = add.clone()
        rc, own, _ = _matmul(a, ta, b, tb, bias, own, out=own)
        assert rc == 0 and torch.equal(own, out[:, :N])


@pytest.mark.parametrize("ta,tb,K", [(0, 0, 64), (0, 1, 512), (1, 1, 520)])
def test_infinities(ta, tb, K):
    announce(f"fp32 product with infinities across {ta} {tb} K{K}")
    gen = torch.Generator().manual_seed(K)
    M = N = 80
    A, Bm = torch.randn(M, K, generator=gen), torch.randn(N, K, generator=gen)
    A[3, 5], A[70, K - 1], A[40, 9] = float("inf"), float("nan"), 3.4e38
    A[41, 2], Bm[7, 2] = 3e30, 3e30  # overflows
    A[42, 2], A[42, 3], Bm[8, 2], Bm[8, 3] = float("inf"), float("inf"), 1.0, -1.0
    want = A @ Bm.t()
    a, b = (A.t().contiguous() if ta else A).cuda(), (Bm.t().contiguous() if tb else Bm).cuda()
    rc, out, _ = _matmul(a, ta, b, tb)
    out = out[:, :N].cpu()
    assert rc == 0
    assert torch.equal(out.isnan(), want.isnan()) and torch.equal(out.isinf(), want.isinf())
    assert torch.equal(out[out.isinf()], want[want.isinf()])
    ok = want.isfinite()
    bound = (K + 36) * EPS * (A.double().abs() @ Bm.double().abs().t())  # (plain fp32 sums, one rounding a step, among them)
    assert ((out.double() - A.double() @ Bm.double().t())[ok].abs() <= bound[ok]).all()


def test_refused():
    a, w = torch.zeros(8, 20, device="cuda"), torch.zeros(8, 20, device="cuda")
    assert _matmul(a, 0, w, 0)[0] == _lib.VIG_ENOTSUP  # a contraction that is no multiple of 8
    assert _matmul(a, 1, w.t().contiguous()[:8], 0)[0] != 0  # both or only the second operand lie across
    flat = torch.zeros(8 * 16 + 1, device="cuda")[1:].view(8, 16)
    assert _matmul(flat, 0, flat, 0)[0] == _lib.VIG_EINVAL
