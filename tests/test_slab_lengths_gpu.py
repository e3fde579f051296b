"""The one-launch forward between 257 tokens and its limit (13 tiles at Dk 64, 16 at Dk 32) and just past it, against the fp64
oracle and the general paths: both forms, views read in place, the fused gate, and what it refuses."""
import ctypes

import pytest
import torch

import vig_amd
from oracle import gla_oracle as O
from vig_amd import _lib, ops
from vig_amd.synthetic import make_gla_inputs, make_locality_weight

from .util import announce, f64, max_abs, oracle_bidir

pytestmark = pytest.mark.gpu

BF16_TOL = 2e-2


def _inputs(B, H, L, Dk, seed, strong=None):
    q, k, v, gf, gb = make_gla_inputs(B, H, L, Dk, 64, seed=seed, dtype=torch.bfloat16)
    if strong is not None:  # gates too strong for the fp16 form in the sequences of the mask
        _, _, _, sf, sb = make_gla_inputs(B, H, L, Dk, 64, seed=seed + 1, dtype=torch.bfloat16, gate_scale=1.0)
        m = strong.reshape(B, H)[:, :, None, None]
        gf, gb = torch.where(m, sf.clamp_min(-3), gf), torch.where(m, sb.clamp_min(-3), gb)
    return [t.cuda() for t in (q, k, v, gf, gb)]


@pytest.mark.parametrize("both", [True, False])
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("L,Dk", [(257, 64), (288, 32), (289, 64), (415, 64), (416, 64), (417, 64), (481, 32), (512, 32), (513, 32)])
def test_lengths(L, Dk, mixed, both):
    announce(f"one-launch lengths L{L} Dk{Dk} mixed={mixed} both={both}")
    B, H = 2, 3
    q, k, v, gf, gb = _inputs(B, H, L, Dk, L, torch.arange(B * H) % 2 == 1 if mixed else None)
    got = vig_amd.gla_bidir_forward(q, k, v, gf, gb if both else None)
    want = oracle_bidir(q, k, v, gf, gb if both else None)
    assert max_abs(f64(got), want) <= BF16_TOL


@pytest.mark.parametrize("B,H,L,Dk", [(2, 6, 300, 32), (1, 3, 512, 32), (3, 2, 416, 64)])
def test_in_place(B, H, L, Dk):
    """Column blocks of a wider matrix, bit for bit the packed call."""
    announce(f"one-launch in place B{B} H{H} L{L} Dk{Dk}")
    q, k, v, gf, gb = _inputs(B, H, L, Dk, 7)
    rows = torch.cat([t.transpose(1, 2).reshape(B, L, -1) for t in (q, k, v)], -1).contiguous()
    ld = rows.shape[-1]
    out = torch.empty_like(v)
    sqk, sv = (ctypes.c_longlong * 3)(L * ld, Dk, ld), (ctypes.c_longlong * 3)(L * ld, 64, ld)
    lib, p = _lib.load(), rows.data_ptr()

    def call(fn, *mid):
        return fn(p, p + 2 * H * Dk, p + 4 * H * Dk, gf.data_ptr(), gb.data_ptr(), *mid)
    s = [ctypes.addressof(x) for x in (sqk, sqk, sv)]
    tail = (Dk ** -0.5, 1.0, 1, 1, ops._stream_ptr(q))
    assert lib.vig_gla_slab_tokens(Dk) >= L
    assert call(lib.vig_gla_slab_fwd, None, out.data_ptr(), B, H, L, Dk, 64, *s, 0, 0, *tail) == _lib.VIG_OK
    assert torch.equal(out, vig_amd.gla_bidir_forward(q, k, v, gf, gb))
    # (the entry point of whole slabs of 256 tokens keeps its limit, the one-launch kernel its own)
    assert call(lib.vig_gla_bidir_fwd_strided, out.data_ptr(), B, H, L, Dk, 64, *s, *tail) == _lib.VIG_ENOTSUP
    assert call(lib.vig_gla_slab_fwd, None, out.data_ptr(), B, H, lib.vig_gla_slab_tokens(Dk) + 1, Dk, 64, *s, 0, 0, *tail) == _lib.VIG_ENOTSUP


@pytest.mark.parametrize("B,H,hw,Dk", [(2, 3, (24, 12), 32), (1, 2, (16, 32), 32), (2, 2, (26, 16), 64), (1, 2, (4, 104), 64),
                                       (1, 2, (3, 126), 64), (1, 1, (32, 16), 64)])
def test_fused_gate(B, H, hw, Dk):
    """The op with the gate in its kernel (or behind it, for grids whose padded rows do not fit) against the two calls."""
    announce(f"one-launch gate B{B} H{H} grid {hw} Dk{Dk}")
    q, k, v, gf, gb = _inputs(B, H, hw[0] * hw[1], Dk, 11)
    w = make_locality_weight(H * 64, 31).cuda()
    got = vig_amd.gla_bidir_locality_gate(q, k, v, gf, gb, w, hw)
    plain = vig_amd.gla_bidir_forward(q, k, v, gf, gb)
    assert torch.equal(got, vig_amd.locality_gate(plain, w, hw))
    want = O.locality_sigmoid_gate_reference(oracle_bidir(q, k, v, gf, gb), f64(w), hw)
    assert max_abs(f64(got), want) <= BF16_TOL


def test_wide_grids_stay_refused():
    q, k, v, gf, gb = _inputs(1, 1, 400, 64, 13)
    with pytest.raises(_lib.VigGlaError):
        vig_amd.gla_bidir_locality_gate(q, k, v, gf, gb, make_locality_weight(64, 31).cuda(), (2, 200))
