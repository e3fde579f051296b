"""fp32 tensors on the matrix cores (gla_f32.hip) against the fp64 oracle, and no less precise than the token-recurrent
fp32 kernel on the same inputs: edges of tiles and segments, one or two directions, gates that leave the tile form's range."""
import numpy as np
import pytest
import torch

import vig_amd
from oracle import gla_oracle as O
from vig_amd.synthetic import make_gla_inputs

from .util import announce, f64, oracle_bidir

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1, 64), (2, 2, 32, 32), (1, 2, 33, 64), (2, 3, 224, 64), (1, 2, 225, 32), (1, 2, 449, 64), (1, 1, 1100, 32)]


@pytest.mark.parametrize("gate_scale", [1 / 16, 1.0, 40.0])  # in range; some tiles beyond it; every tile beyond it
@pytest.mark.parametrize("B,H,L,Dk", SHAPES)
def test_forward(B, H, L, Dk, gate_scale):
    announce(f"fp32 forward on the matrix cores B{B} H{H} L={L} Dk={Dk} gates x {gate_scale}")
    t = make_gla_inputs(B, H, L, Dk, 64, seed=900 + L, dtype=torch.float32, gate_scale=gate_scale)
    for args in (t, (*t[:4], None)):
        want = oracle_bidir(*args)
        x = [a.cuda() if a is not None else None for a in args]
        err = lambda o: np.linalg.norm(f64(o) - want) / np.linalg.norm(want)
        mine, serial = err(vig_amd.gla_bidir_forward(*x)), err(vig_amd.gla_bidir_forward(*x, exact=True))
        print(f"  relative error {mine:.2e}, token-recurrent {serial:.2e}", flush=True)
        assert mine <= max(2 * serial, 3e-7)


# what leaves the range of the common form, in one direction or both, and how: a whole tile's gates, one channel's, single tokens
# (on both sides of every level's split), and what the form for any gates does not take either: gates that grow, no numbers
@pytest.mark.parametrize("kind", ["one tile", "one channel", "tokens", "infinite", "reverse only", "growing", "growing a little"])
@pytest.mark.parametrize("L,Dk", [(31, 64), (64, 32), (197, 64), (224, 32), (450, 64)])
def test_forward_beyond_the_range(L, Dk, kind):
    announce(f"fp32 forward, gates beyond the range: {kind}, L={L} Dk={Dk}")
    q, k, v, gf, gb = make_gla_inputs(1, 3, L, Dk, 64, seed=300 + L, dtype=torch.float32)
    if kind == "one tile":
        gf[0, 1, L // 2:L // 2 + 20] -= 3.0
    elif kind == "one channel":
        gf[0, :, :, 5] -= 2.0
        gb[0, :, :, Dk - 1] -= 5.0
    elif kind == "tokens":
        for t in (0, 1, 3, 7, 15, 16, 30):
            gf[0, :, t::32] -= 9.0
            gb[0, :, (31 - t)::32] -= 9.0
    elif kind == "infinite":
        gf[0, :, 3::5, 1::3] = -float("inf")
        gb[0, :, 2::9] = -float("inf")
    elif kind == "reverse only":
        gb[0, 0] -= 1.5
    else:
        gf[0, 1] -= 1.5
        gf[0, 1, 4:9, 3] = 0.5 if kind == "growing a little" else 2.0
    for args in ((q, k, v, gf, gb), (q, k, v, gf, None)):
        want = oracle_bidir(*args)
        x = [a.cuda() if a is not None else None for a in args]
        err = lambda o: np.linalg.norm(f64(o) - want) / np.linalg.norm(want)
        mine, serial = err(vig_amd.gla_bidir_forward(*x)), err(vig_amd.gla_bidir_forward(*x, exact=True))
        print(f"  relative error {mine:.2e}, token-recurrent {serial:.2e}", flush=True)
        assert mine <= max(2 * serial, 3e-7)
    gf[0, 2, 1, 2] = float("nan")
    got = f64(vig_amd.gla_bidir_forward(q.cuda(), k.cuda(), v.cuda(), gf.cuda()))
    assert np.isnan(got[0, 2, 1]).all() and np.isfinite(got[0, 0, :]).all()


def test_forward_magnitudes_and_infinite_gates():
    """Inputs beyond the tile form's magnitude bound take the serial form, gates of -inf the form for any gates."""
    announce("fp32 forward, large magnitudes and gates of -inf")
    q, k, v, gf, gb = make_gla_inputs(1, 2, 300, 64, 64, seed=5, dtype=torch.float32)
    q[0, 0, 3] *= 1e14
    gf[0, 1, 40:60:7] = -float("inf")
    want = oracle_bidir(q, k, v, gf, gb)
    got = f64(vig_amd.gla_bidir_forward(*(t.cuda() for t in (q, k, v, gf, gb))))
    for h in range(2):
        assert np.abs(got[0, h] - want[0, h]).max() <= 1e-5 * np.abs(want[0, h]).max()


@pytest.mark.parametrize("gate_scale", [1 / 16, 1.0])  # in range; beyond it (flagged for the recurrent kernel)
@pytest.mark.parametrize("B,H,L,Dk", [(1, 1, 2, 64), (2, 2, 33, 32), (2, 3, 196, 32), (1, 2, 224, 64), (1, 2, 225, 64),
                                      (1, 2, 256, 32), (1, 2, 449, 64), (1, 1, 700, 32),
                                      (1, 769, 5, 64), (1, 768, 16, 64), (2, 1, 17, 64)])
def test_backward(B, H, L, Dk, gate_scale):
    announce(f"fp32 backward on the matrix cores B{B} H{H} L={L} Dk={Dk} gates x {gate_scale}")
    t = make_gla_inputs(B, H, L, Dk, 64, seed=950 + L, dtype=torch.float32, gate_scale=gate_scale)
    d_o = torch.randn(t[2].shape, generator=torch.Generator().manual_seed(4))
    for args in (t, (*t[:4], None)):
        want = O.bidir_gla_backward(*(f64(a) if a is not None else None for a in args), f64(d_o), out_scale=0.5)
        x = [a.cuda() if a is not None else None for a in (*args, d_o)]
        mine = vig_amd.gla_bidir_backward(*x, out_scale=0.5)
        serial = vig_amd.gla_bidir_backward(*x, out_scale=0.5, exact=True)
        for name, a, b, w in zip(("dq", "dk", "dv", "dg_fwd", "dg_bwd"), mine, serial, want):
            if w is None:
                assert a is None
                continue
            err = lambda y: np.linalg.norm(f64(y) - w) / np.linalg.norm(w)
            assert err(a) <= max(2 * err(b), 4e-7), (name, err(a), err(b))


# some sequences flagged for the recurrent kernel, whose two directions then run side by side, among others that are not
@pytest.mark.parametrize("B,H,L,Dk", [(2, 3, 17, 32), (3, 7, 197, 64), (1, 5, 450, 32)])
def test_backward_of_some_sequences_beyond_the_range(B, H, L, Dk):
    announce(f"fp32 backward, every third sequence beyond the range, B{B} H{H} L={L} Dk={Dk}")
    t = make_gla_inputs(B, H, L, Dk, 64, seed=970 + L, dtype=torch.float32)
    for g in t[3:]:
        g.view(B * H, L, Dk)[::3] -= 2.5
    d_o = torch.randn(t[2].shape, generator=torch.Generator().manual_seed(5))
    want = O.bidir_gla_backward(*(f64(a) for a in t), f64(d_o), out_scale=0.5)
    x = [a.cuda() for a in (*t, d_o)]
    mine = vig_amd.gla_bidir_backward(*x, out_scale=0.5)
    serial = vig_amd.gla_bidir_backward(*x, out_scale=0.5, exact=True)
    for name, a, b, w in zip(("dq", "dk", "dv", "dg_fwd", "dg_bwd"), mine, serial, want):
        flat = w.reshape(B * H, -1)
        err = lambda y: np.linalg.norm(f64(y).reshape(B * H, -1) - flat, axis=1) / np.linalg.norm(flat, axis=1)
        assert (err(a) <= np.maximum(2 * err(b), 4e-7)).all(), (name, err(a), err(b))
        assert torch.equal(a.view(B * H, L, -1)[::3], b.view(B * H, L, -1)[::3]), name  # (the same sums, whichever direction ends first)
    for _ in range(5):
        assert all(torch.equal(a, b) for a, b in zip(mine, vig_amd.gla_bidir_backward(*x, out_scale=0.5)))
