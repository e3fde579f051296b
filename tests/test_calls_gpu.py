"""The native op-level calls (csrc/py_calls.cpp) against the ctypes binding they stand in front of."""
import pytest
import torch

import vig_amd
from vig_amd import _ext, ops
from vig_amd.synthetic import make_gla_inputs, make_locality_weight

from .util import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,L,Dk,Dv,dtype", [(1, 1, 1, 32, 64, torch.bfloat16), (2, 3, 257, 64, 64, torch.bfloat16),
                                               (2, 2, 130, 16, 32, torch.bfloat16), (2, 2, 33, 64, 32, torch.float32)])
def test_calls_match_ctypes(monkeypatch, B, H, L, Dk, Dv, dtype):
    announce(f"native calls B{B} H{H} L={L} Dk={Dk} Dv={Dv} {dtype}")
    assert _ext.calls() is not None
    q, k, v, gf, gb = (t.cuda() for t in make_gla_inputs(B, H, L, Dk, Dv, seed=3, dtype=dtype))
    g = torch.cat([gf, gb])
    d_o = torch.randn_like(v)
    w = make_locality_weight(H * Dv, seed=7).cuda()

    def everything():
        out = [vig_amd.gla_bidir_locality_gate(q, k, v, gf, gb, w, (L, 1))]
        for f, x in ((lambda *a: vig_amd.batch_bid_fused_chunk_gla(*a)[0], (q, k, v, g)), (ops.gla_bidir_forward, (q, k, v, gf, gb)),
                     (ops.gla_bidir_forward, (q, k, v, gf)), (lambda *a: ops.gla_bidir_forward(*a, exact=True), (q, k, v, gf, gb))):
            leaves = [t.clone().requires_grad_() for t in x]
            o = f(*leaves)
            out += [f(*x), o.detach(), *torch.autograd.grad(o, leaves, d_o)]
        return out

    got = everything()
    with monkeypatch.context() as m:
        m.setattr(_ext, "calls", lambda: None)
        want = everything()
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and torch.equal(a, b)
    # a view takes the general path, with the same values
    qt = q.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(ops.gla_bidir_forward(qt, k, v, gf, gb), ops.gla_bidir_forward(q, k, v, gf, gb))
