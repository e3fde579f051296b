"""The locality gate inside the op's kernel against the two calls, bit for bit, where outputs of the op are beyond fp16's range, below its grid,
around its limits, zero, or large enough for the sigmoid's tail, and at every length the kernel takes."""
import pytest
import torch

import vig_amd
from vig_amd.synthetic import make_gla_inputs, make_locality_weight

from .util import announce

pytestmark = pytest.mark.gpu

# factors of q, k, v in every second head: fp16 form with outputs beyond 65504, general form, outputs below 2^-17, both ends in one slab
RANGES = {"large": (20.0, 8.0, 800.0), "huge": (1.0, 1.0, 2.0 ** 40), "small": (1.0, 1.0, 2.0 ** -24), "mixed": None}


@pytest.mark.parametrize("what", RANGES)
@pytest.mark.parametrize("hw,Dk", [((1, 1), 64), ((7, 7), 32), ((14, 14), 64), ((16, 16), 32), ((16, 17), 64), ((20, 20), 32), ((26, 16), 64),
                                   ((16, 32), 32)])
def test_equals_two_calls(hw, Dk, what):
    announce(f"gate range {what} grid {hw} Dk{Dk}")
    B, H, L = 2, 4, hw[0] * hw[1]
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, L, Dk, 64, seed=L + Dk, dtype=torch.bfloat16))
    if what == "mixed":
        v[:, 1::2, ::3] *= 2.0 ** -24
        v[:, 1::2, 1::5] *= 1000.0
        q[:, 1::2] *= 20.0
        k[:, 1::2] *= 8.0
    else:
        for t, f in zip((q, k, v), RANGES[what]):
            t[:, 1::2] *= f
    w = make_locality_weight(H * 64, 31).cuda()
    plain = vig_amd.gla_bidir_forward(q, k, v, gf, gb)
    assert torch.isfinite(plain).all()
    if what in ("large", "huge"):
        assert (plain.abs() > 65504).any() or L == 1
    want = vig_amd.locality_gate(plain, w, hw)
    got = vig_amd.gla_bidir_locality_gate(q, k, v, gf, gb, w, hw)
    assert torch.isfinite(got).all()
    assert torch.equal(got, want)


@pytest.mark.parametrize("top", [0.0, 2.0 ** -23, 300.0, 500.0, 1020.0, 1024.0, 65000.0])
@pytest.mark.parametrize("Dk", [32, 64])
def test_largest_output(Dk, top):
    """All outputs scaled to a largest one; 0: a head without values, a channel without, a masked query."""
    announce(f"gate range, largest output {top} Dk{Dk}")
    B, H, hw = 2, 3, (14, 14)
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, 196, Dk, 64, seed=3, dtype=torch.bfloat16))
    if top == 0:
        v[:, 1], v[:, :, :, 5], q[:, :, 7] = 0, 0, 0
    factor = top / float(vig_amd.gla_bidir_forward(q, k, v, gf, gb).float().abs().max()) if top else 1.0
    w = make_locality_weight(H * 64, 31).cuda()
    want = vig_amd.locality_gate(vig_amd.gla_bidir_forward(q, k, v, gf, gb, -1, factor), w, hw)
    assert torch.equal(vig_amd.gla_bidir_locality_gate(q, k, v, gf, gb, w, hw, -1, factor), want)
