"""fp32 on the matrix cores, sequences longer than one workgroup takes: as many short segments as fill the chip, segments of seven
tiles for many sequences or little room; forward and backward against fp64, one and both directions."""
import pytest
import torch

import vig_amd
from oracle import gla_oracle as O
from vig_amd import _lib, ops
from vig_amd.synthetic import make_gla_inputs

from .test_backward_gpu import _check_all, _do
from .util import announce, f64, max_rel, oracle_bidir

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("both", [True, False])
@pytest.mark.parametrize("B,H,L,Dk", [(1, 2, 225, 32), (1, 2, 225, 64), (1, 1, 257, 64), (1, 3, 289, 32), (1, 2, 449, 64), (3, 1, 260, 32)])
def test_few_sequences(B, H, L, Dk, both):
    announce(f"fp32 segments B{B} H{H} L{L} Dk{Dk} both={both}")
    q, k, v, gf, gb = make_gla_inputs(B, H, L, Dk, 64, seed=L)
    gb = gb if both else None
    do = _do(v.shape, 2, torch.float32)
    dev = [None if t is None else t.cuda() for t in (q, k, v, gf, gb)]
    assert max_rel(f64(vig_amd.gla_bidir_forward(*dev)), oracle_bidir(q, k, v, gf, gb)) <= 1e-5
    got = vig_amd.gla_bidir_backward(*dev, do.cuda(), out_scale=0.5 if both else 1.0)
    if both:
        want = O.bidir_gla_backward(f64(q), f64(k), f64(v), f64(gf), f64(gb), f64(do), out_scale=0.5)
    else:
        want = [*O.gla_recurrent_backward(f64(q), f64(k), f64(v), f64(gf), f64(do)), None]
    _check_all(got, want, q, tol=1e-5)


@pytest.mark.parametrize("B,H,L,Dk", [(40, 6, 230, 32), (50, 3, 300, 64)])
def test_many_sequences(B, H, L, Dk):
    announce(f"fp32 segments, {B * H} sequences of {L}, Dk{Dk}")
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, L, Dk, 64, seed=3))
    do = _do(v.shape, 4, torch.float32).cuda()
    assert max_rel(f64(vig_amd.gla_bidir_forward(q, k, v, gf, gb)), f64(vig_amd.gla_bidir_forward(q, k, v, gf, gb, exact=True))) <= 1e-5
    want = vig_amd.gla_bidir_backward(q, k, v, gf, gb, do, exact=True)
    _check_all(vig_amd.gla_bidir_backward(q, k, v, gf, gb, do), [f64(t) for t in want], q.cpu(), tol=1e-5)


def test_workspace_of_seven_tile_segments():
    """A caller with room for segments of seven tiles only is still served on the matrix cores."""
    lib, B, H, L, Dk = _lib.load(), 1, 3, 700, 32
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, L, Dk, 64, seed=8))
    slots = 2 * 4160 * 4  # both directions of one segment
    need = lib.vig_gla_bidir_fwd_workspace_for(B, H, L, Dk, 64, 0, 0, 1)
    assert need == B * H * 11 * slots  # 22 tiles by two
    outs = []
    for n in (need, B * H * 4 * slots):
        ws, o = torch.empty(n, dtype=torch.uint8, device="cuda"), torch.empty_like(v)
        rc = lib.vig_gla_bidir_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), gf.data_ptr(), gb.data_ptr(), o.data_ptr(), ws.data_ptr(), n,
                                   B, H, L, Dk, 64, Dk ** -0.5, 1.0, 0, 0, ops._stream_ptr(q))
        assert rc == _lib.VIG_OK
        outs.append(o)
    want = oracle_bidir(*(t.cpu() for t in (q, k, v, gf, gb)))
    assert all(max_rel(f64(o), want) <= 1e-5 for o in outs) and not torch.equal(*outs)
