"""The op that makes its gates from rank-16 rows and reads q, k, v in place, against the gate kernel, packed tensors and the op: edges of
tiles and segments, one token, several heads and images, clamps, gates too strong for the fp16 form, and what it refuses."""
import ctypes

import pytest
import torch

import vig_amd
from vig_amd import _lib, ops

from .util import announce

pytestmark = pytest.mark.gpu


def _run(z, w, b, B, H, L, clamp, inv_norm=1 / 16, Dk=32, short=0):
    ld, n = z.shape[-1], H * (2 * Dk + 64)
    lib, p, tail = _lib.load(), z.data_ptr(), (Dk ** -0.5, 1.0)
    s = [(ctypes.c_longlong * 3)(L * ld, d, ld) for d in (Dk, Dk, 64)]
    st = [ctypes.addressof(x) for x in s]
    low = p + 2 * (n + H * 64)
    out = torch.empty(B, H, L, 64, dtype=z.dtype, device="cuda")
    need = lib.vig_gla_lowrank_fwd_workspace(B, H, L, Dk, 64)
    ws = torch.full((need + 256,), 77, dtype=torch.uint8, device="cuda")
    rc = lib.vig_gla_lowrank_fwd(p, p + 2 * H * Dk, p + 4 * H * Dk, low, ld, w.data_ptr(), b.data_ptr(), out.data_ptr(), ws.data_ptr(),
                                 need - short, B, H, L, Dk, 64, *st, inv_norm, clamp, *tail, 1, ops._stream_ptr(z))
    assert (ws[need:] == 77).all()
    if rc != _lib.VIG_OK:
        return rc, None, None
    gates = torch.empty(2, B, H, L, Dk, dtype=z.dtype, device="cuda")
    assert lib.vig_dirgate_lowrank_fwd(low, ld, w.data_ptr(), b.data_ptr(), gates.data_ptr(), B, L, H, Dk, 16, inv_norm, clamp, 1, 1,
                                       ops._stream_ptr(z)) == _lib.VIG_OK
    q, k, v = (z[..., i:i + H * d].reshape(B, L, H, d).transpose(1, 2).contiguous() for i, d in ((0, Dk), (H * Dk, Dk), (2 * H * Dk, 64)))
    return rc, out, vig_amd.gla_bidir_forward(q, k, v, gates[0], gates[1], scale=Dk ** -0.5)


def _inputs(B, H, L, seed, strength=1.0, Dk=32):
    gen = torch.Generator().manual_seed(seed)
    z = torch.randn(B, L, H * (2 * Dk + 128) + 32, generator=gen).bfloat16().cuda()
    w, b = torch.randn(2 * H * Dk, 16, generator=gen) * 0.25 * strength, torch.randn(2 * H * Dk, generator=gen) * strength
    return z, w.bfloat16().cuda(), b.bfloat16().cuda()


@pytest.mark.parametrize("B,H,L", [(1, 1, 1), (2, 3, 31), (1, 2, 33), (3, 3, 196), (2, 6, 225), (1, 2, 320), (1, 3, 512), (2, 1, 481),
                                   (1, 1, 513), (2, 3, 784), (1, 2, 897), (1, 3, 2305)])
@pytest.mark.parametrize("clamp", [float("nan"), -0.05])
def test_against_separate_launches(B, H, L, clamp):
    announce(f"gates in the op B{B} H{H} L{L} clamp {clamp}")
    rc, got, want = _run(*_inputs(B, H, L, L), B, H, L, clamp)
    assert rc == _lib.VIG_OK and torch.equal(got, want)


@pytest.mark.parametrize("L", [45, 196, 300, 700])
def test_strong_gates(L):
    announce(f"gates in the op, general form L{L}")
    rc, got, want = _run(*_inputs(2, 3, L, 5, strength=4.0), 2, 3, L, float("nan"), inv_norm=1.0)
    assert rc == _lib.VIG_OK and torch.equal(got, want)


def test_refused():
    z, w, b = _inputs(1, 1, 513, 3)
    assert _run(z, w, b, 1, 1, 513, float("nan"), short=4)[0] == _lib.VIG_ENOSPC
    z, w, b = _inputs(1, 1, 64, 3, Dk=64)
    assert _run(z, w, b, 1, 1, 64, float("nan"), Dk=64)[0] == _lib.VIG_ENOTSUP
