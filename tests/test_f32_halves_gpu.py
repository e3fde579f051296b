"""The fp32 backward with the two directions of what fills less than half the chip in workgroups of their own, against the fp64 oracle and
against the call that has no room for it: whole sequences and segments, leftovers of full rounds, flagged sequences."""
import pytest
import torch

from oracle import gla_oracle as O
from vig_amd import _lib
from vig_amd.synthetic import make_gla_inputs

from .test_backward_gpu import _check_all
from .util import announce, f64

pytestmark = pytest.mark.gpu


def _run(q, k, v, gf, gb, do, size):
    B, H, L, Dk = q.shape
    out = [torch.empty_like(t) for t in (q, k, v, gf, gb)]
    ws = torch.full((size + 512,), 77, dtype=torch.uint8, device="cuda")
    rc = _lib.load().vig_gla_bidir_bwd(*(t.data_ptr() for t in (q, k, v, gf, gb, do, *out)), ws.data_ptr(), size, B, H, L, Dk, 64, Dk ** -0.5,
                                       1.0, 0, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.VIG_OK and (ws[size:] == 77).all()
    return out


@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("Dk", [32, 64])
@pytest.mark.parametrize("B,H,L", [(1, 1, 33), (3, 2, 196), (2, 2, 224), (2, 3, 400), (1, 2, 1090), (130, 2, 200), (129, 3, 40)])
def test_against_oracle(B, H, L, Dk, strong):
    announce(f"fp32 halves B{B} H{H} L{L} Dk{Dk} strong={strong}")
    q, k, v, gf, gb = make_gla_inputs(B, H, L, Dk, 64, seed=L, dtype=torch.float32)
    if strong:  # some sequences out of the tile form's range: the recurrent kernel does them
        _, _, _, sf, _ = make_gla_inputs(B, H, L, Dk, 64, seed=L + 1, dtype=torch.float32, gate_scale=1.0)
        m = (torch.arange(B * H) % 3 == 1).reshape(B, H)[:, :, None, None]
        gf = torch.where(m, 3 * sf, gf)
    do = torch.randn(v.shape, generator=torch.Generator().manual_seed(L))
    t = [x.cuda() for x in (q, k, v, gf, gb, do)]
    lib = _lib.load()
    most = lib.vig_gla_bidir_bwd_workspace_for(B, H, L, Dk, 64, 0, 0, 1)
    least = lib.vig_gla_bidir_bwd_workspace(B, H, L, Dk, 64, 1)
    got = _run(*t, most)
    pick = sorted({0, B // 2, B - 1})
    want = O.bidir_gla_backward(*(f64(x[pick]) for x in t))
    _check_all([a[pick] for a in got], want, q[pick], tol=1e-5)
    if least < most:  # without room for halves: the same sums in another order
        _check_all(_run(*t, least), [f64(a) for a in got], q, tol=1e-5)

