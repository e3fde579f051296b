"""Sums over partial rows that several backward kernels put off and one launch makes, against each of them on its own: few and many rows, a bias gradient
off the 16-byte boundary, a full list."""
import ctypes

import pytest
import torch

from vig_amd import _lib

from .util import announce

pytestmark = pytest.mark.gpu


class _Jobs(ctypes.Structure):
    _fields_ = [("job", ctypes.c_char * (32 * 12)), ("count", ctypes.c_int)]


@pytest.mark.parametrize("B,h,w,H", [(1, 3, 5, 1), (3, 14, 14, 3), (130, 14, 14, 6)])
def test_against_separate_sums(B, h, w, H):
    announce(f"sums put off B{B} {h}x{w} C{64 * H}")
    g = torch.Generator(device="cuda").manual_seed(B)
    L, C, rows = h * w, 64 * H, B * h * w
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    f = lambda *s: torch.empty(*s, device="cuda")  # noqa: E731
    x, dy, o, glin = r(rows, C), r(rows, C), r(B, H, L, 64), r(rows, C)
    nw, wg, taps = torch.rand(C, generator=g, device="cuda"), torch.rand(64, generator=g, device="cuda"), torch.randn(C, 9, generator=g, device="cuda")
    p, lib, st = (lambda t: t.data_ptr()), _lib.load(), torch.cuda.current_stream().cuda_stream
    ws = [torch.empty(n, dtype=torch.uint8, device="cuda") for n in (lib.vig_rmsnorm_bwd_workspace(rows, C), lib.vig_locality_blend_bwd_workspace(B, L, 64),
                                                                     lib.vig_dwconv3x3_bwd_weight_workspace(B, C))]
    ints = lambda *v: (ctypes.c_int * 2)(*v)  # noqa: E731
    ptrs = lambda *v: (ctypes.c_void_p * 2)(*v)  # noqa: E731
    longs = lambda *v: (ctypes.c_longlong * 2)(*v)  # noqa: E731
    N, K = ints(C, C), ints(C, 64)
    ws.append(torch.empty(lib.vig_linear_bwd_weight_many_workspace(rows, N, K, 2), dtype=torch.uint8, device="cuda"))

    def run(later):
        out = [f(C), f(128), f(10 * C), f(C, C), f(C, 64), f(C + 1)]
        tail, name = ([ctypes.byref(later)], "_later") if later is not None else ([], "")
        scratch = [torch.empty_like(x) for _ in range(5)]
        call = lambda fn, *a: getattr(lib, fn + name)(*a, *tail, st)  # noqa: E731
        if later is not None:  # (the list goes in front of the stream)
            call = lambda fn, *a: getattr(lib, fn + name)(*a, ctypes.byref(later), st)  # noqa: E731
        assert call("vig_rmsnorm_mixed_bwd", p(x), p(nw), p(dy), None, p(scratch[0]), None, p(out[0]), p(ws[0]), ws[0].numel(), rows, C, 1e-5, 1, 1) == 0
        assert call("vig_locality_blend_bwd_strided", p(o), p(x), p(glin), p(wg), p(wg), p(dy), p(scratch[1]), p(scratch[2]), p(scratch[3]), p(out[1]),
                    p(ws[1]), ws[1].numel(), B, H, L, 64, C, C, 1e-5, 1, 1) == 0
        assert call("vig_dwconv3x3_bwd", p(x), p(dy), None, p(taps), p(scratch[4]), p(out[2]), p(ws[2]), ws[2].numel(), B, h, w, C, 1) == 0
        assert call("vig_linear_bwd_weight_many", ptrs(p(dy), p(dy)), longs(C, C), ptrs(p(x), p(x)), longs(C, C), ptrs(p(out[3]), p(out[4])),
                    ptrs(None, p(out[5]) + 4), p(ws[3]), ws[3].numel(), rows, N, K, 2) == 0
        if later is not None:
            assert lib.vig_sum_jobs_run(ctypes.byref(later), st) == 0 and later.count == 0
        return out[:5] + [out[5][1:]]

    want, got = run(None), run(_Jobs())
    assert all(torch.equal(a, b) for a, b in zip(got, want))  # the same sums in the same order


def test_refused():
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    x, w, out = torch.zeros(8, 64, dtype=torch.bfloat16, device="cuda"), torch.ones(64, device="cuda"), torch.zeros(64, device="cuda")
    ws, jobs = torch.empty(lib.vig_rmsnorm_bwd_workspace(8, 64), dtype=torch.uint8, device="cuda"), _Jobs()
    call = lambda: lib.vig_rmsnorm_mixed_bwd_later(x.data_ptr(), w.data_ptr(), x.data_ptr(), None, torch.empty_like(x).data_ptr(), None, out.data_ptr(),  # noqa: E731
                                                   ws.data_ptr(), ws.numel(), 8, 64, 1e-5, 1, 1, ctypes.byref(jobs), st)
    assert all(call() == _lib.VIG_OK for _ in range(12)) and call() == _lib.VIG_EINVAL  # the list is full
    assert lib.vig_sum_jobs_run(ctypes.byref(jobs), st) == _lib.VIG_OK and jobs.count == 0
    jobs.count = 13
    assert call() == _lib.VIG_EINVAL and lib.vig_sum_jobs_run(ctypes.byref(jobs), st) == _lib.VIG_EINVAL
    assert lib.vig_sum_jobs_run(None, st) == _lib.VIG_EINVAL
