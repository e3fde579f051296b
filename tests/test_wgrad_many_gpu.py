"""Weight and bias gradients of several layers over the same rows in one launch, against float64 products."""
import ctypes

import pytest
import torch

from vig_amd import _lib

pytestmark = pytest.mark.gpu
LAYERS = [(128, 128, True), (384, 16, True), (136, 264, False), (8, 8, True)]  # whole tiles, narrow, remainders, the least


def _call(dys, xs, biases):
    lib, n = _lib.load(), len(dys)
    arr = lambda t, v: (t * n)(*v)  # noqa: E731
    T, N, K = dys[0].shape[0], [d.shape[1] for d in dys], [x.shape[1] for x in xs]
    dw = [torch.full((a, b), float("nan"), device="cuda") for a, b in zip(N, K)]
    db = [torch.full((a,), float("nan"), device="cuda") if w else None for a, w in zip(N, biases)]
    cN, cK = arr(ctypes.c_int, N), arr(ctypes.c_int, K)
    need = lib.vig_linear_bwd_weight_many_workspace(T, cN, cK, n)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    rc = lib.vig_linear_bwd_weight_many(
        arr(ctypes.c_void_p, [d.data_ptr() for d in dys]), arr(ctypes.c_longlong, [d.stride(0) for d in dys]),
        arr(ctypes.c_void_p, [x.data_ptr() for x in xs]), arr(ctypes.c_longlong, [x.stride(0) for x in xs]),
        arr(ctypes.c_void_p, [w.data_ptr() for w in dw]), arr(ctypes.c_void_p, [b.data_ptr() if b is not None else None for b in db]),
        ws.data_ptr(), need, T, cN, cK, n, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return dw, db


def _check(dys, xs, dw, db):
    for d, x, w, b in zip(dys, xs, dw, db):
        # sums of T fp32 products, each exact: at most T roundings of 2^-24 of the running sum of magnitudes
        bound = d.shape[0] * 2.0 ** -24
        d, x = d.double(), x.double()
        assert ((w.double() - d.t() @ x).abs() <= bound * (d.abs().t() @ x.abs()) + 1e-30).all()
        if b is not None:
            assert ((b.double() - d.sum(0)).abs() <= bound * d.abs().sum(0) + 1e-30).all()


@pytest.mark.parametrize("T", [1, 31, 33, 256, 257, 1571])  # one row, around a stage, one and several ranges with a rest
@pytest.mark.parametrize("count", [1, 2, 4])
def test_layers_together(T, count):
    g = torch.Generator("cuda").manual_seed(T + count)
    r = lambda n: torch.randn(T, n + 24, device="cuda", generator=g).bfloat16()[:, 8:8 + n]  # (columns of wider rows)  # noqa: E731
    layers = LAYERS[-count:]
    dys, xs = [r(n) for n, _, _ in layers], [r(k) for _, k, _ in layers]
    if T == 1:  # (torch reports any stride for a single row)
        dys, xs = [d.contiguous() for d in dys], [x.contiguous() for x in xs]
    _check(dys, xs, *_call(dys, xs, [b for _, _, b in layers]))


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("T", [20, 700])  # one range; several, whose partial sums are added
@pytest.mark.parametrize("N", [8, 48, 136, 384])  # a part of a block of 32 channels, one and a half, a tile and a rest, whole tiles
def test_a_channel_keeps_to_itself(N, T, value):
    """Gradients that overflowed in one channel leave every other channel's sums bit for bit what they are without it."""
    g = torch.Generator("cuda").manual_seed(N + T)
    dy, x = (torch.randn(T, n, device="cuda", generator=g).bfloat16() for n in (N, 40))
    (dw0,), (db0,) = _call([dy], [x], [True])
    for n in sorted({0, 7, N // 2, N - 8, N - 1}):
        bad = dy.clone()
        bad[T // 3, n] = value
        (dw,), (db,) = _call([bad], [x], [True])
        others = torch.arange(N, device="cuda") != n
        assert torch.equal(db[others], db0[others]) and torch.equal(dw[others], dw0[others])
        assert torch.equal(db[n].nan_to_num(nan=7.0), torch.tensor(value, device="cuda").nan_to_num(nan=7.0))
        assert not dw[n].isfinite().any()


@pytest.mark.parametrize("T", [16384, 16385])  # 274 tiles: in one launch, and a layer behind the other
def test_many_tiles(T):
    g = torch.Generator("cuda").manual_seed(T)
    dys, xs = zip(*([torch.randn(T, n, device="cuda", generator=g).bfloat16() for n in nk] for nk in ((2048, 2056), (136, 24))))
    _check(dys, xs, *_call(dys, xs, [True, True]))


def test_rows_far_apart():  # past 32-bit byte offsets inside a stage
    T, ld, n, k = 40, (1 << 26) + 8, 136, 24
    dy = torch.empty(T * ld, dtype=torch.bfloat16, device="cuda").as_strided((T, n), (ld, 1))
    dy.copy_(torch.randn(T, n, device="cuda"))
    x = torch.randn(T, k, device="cuda").bfloat16()
    _check([dy], [x], *_call([dy], [x], [True]))


def test_refusals_and_the_single_call():
    lib = _lib.load()
    one = (ctypes.c_int * 5)(*[64] * 5)
    assert lib.vig_linear_bwd_weight_many_workspace(100, one, one, 5) == 0
    assert lib.vig_linear_bwd_weight_many_workspace(100, one, one, 0) == 0
    assert lib.vig_linear_bwd_weight_many_workspace(100, one, one, 1) == lib.vig_linear_bwd_weight_workspace(100, 64, 64) > 0
    assert lib.vig_linear_bwd_weight_many(None, None, None, None, None, None, None, 0, 100, one, one, 1, None) < 0
