"""vig_gla_lowrank_fwd past the one-launch kernel's length: what it refuses before any launch, and plain tensors given as token stride 0."""
import ctypes

import pytest
import torch

from vig_amd import _lib


def _strides(*s):
    return (ctypes.c_longlong * 3)(*s)


def _call(lib, pointers, o, ws, B, H, L, sq, sk, sv, stream=None):
    q, k, v, low, w, b = pointers
    need = lib.vig_gla_lowrank_fwd_workspace(B, H, L, 32, 64)
    return lib.vig_gla_lowrank_fwd(q, k, v, low, 16, w, b, o, ws, need, B, H, L, 32, 64, *(ctypes.addressof(x) for x in (sq, sk, sv)),
                                   1 / 16, float("nan"), 32 ** -0.5, 1.0, _lib.VIG_BF16, stream)


@pytest.mark.skipif(torch.cuda.is_available(), reason="pointers to nothing: only where no launch can follow")
def test_refused_before_any_launch():
    lib, L = _lib.load(), 600
    p = [4096] * 6
    qk, v = _strides(L * 32, L * 32, 32), _strides(L * 64, L * 64, 64)
    # as many sequences and directions as the scan's grid holds are launched (and fail here for want of a device)
    assert _call(lib, p, 4096, 4096, 32767, 1, L, qk, qk, v) not in (_lib.VIG_ENOTSUP, _lib.VIG_EINVAL)
    assert _call(lib, p, 4096, 4096, 32768, 1, L, qk, qk, v) == _lib.VIG_ENOTSUP
    assert _call(lib, p, 4096, 4096, 8192, 5, L, qk, qk, v) == _lib.VIG_ENOTSUP
    for bad in (_strides(L * 32, L * 32, 36), _strides(L * 32, -32, 32), _strides(0, 32, 32), _strides(L << 21, 32, 1 << 21)):
        assert _call(lib, p, 4096, 4096, 2, 3, L, qk, bad, v) == _lib.VIG_EINVAL
        assert _call(lib, p, 4096, 4096, 2, 3, L, qk, qk, bad) == _lib.VIG_EINVAL
        assert _call(lib, p, 4096, 4096, 2, 3, L, bad, qk, v) == _lib.VIG_EINVAL


@pytest.mark.gpu
@pytest.mark.parametrize("L", [300, 600])
def test_token_stride_zero_is_plain(L):
    print(f"[case] low-rank op, plain tensors as token stride 0, L{L}", flush=True)
    lib, B, H = _lib.load(), 2, 3
    gen = torch.Generator().manual_seed(L)
    r = lambda *s: torch.randn(*s, generator=gen).bfloat16().cuda()  # noqa: E731
    t = [r(B, H, L, 32), r(B, H, L, 32), r(B, H, L, 64), r(B, L, 16), r(2 * H * 32, 16), r(2 * H * 32)]
    p = [x.data_ptr() for x in t]
    need = lib.vig_gla_lowrank_fwd_workspace(B, H, L, 32, 64)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    qk, v, none = _strides(H * L * 32, L * 32, 32), _strides(H * L * 64, L * 64, 64), _strides(0, 0, 0)
    out = []
    for s in ((qk, qk, v), (none, none, none), (qk, none, v), (qk, qk, none)):
        out.append(torch.full_like(t[2], float("nan")))
        assert _call(lib, p, out[-1].data_ptr(), ws.data_ptr(), B, H, L, *s, torch.cuda.current_stream().cuda_stream) == _lib.VIG_OK
    assert torch.isfinite(out[0]).all() and all(torch.equal(o, out[0]) for o in out[1:])
