"""The fp32 forward and backward with the two directions of what fills less than half the chip in workgroups of their own, against the fp64 oracle and
against the call that has no room for it: whole sequences and segments, leftovers of full rounds, flagged sequences."""
import pytest
import torch

from oracle import gla_oracle as O
from vig_amd import _lib
from vig_amd.synthetic import make_gla_inputs

from .test_backward_gpu import _check_all
from .util import announce, f64, max_rel, oracle_bidir

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



@pytest.mark.parametrize("gates", ["mild", "strong", "positive"])
@pytest.mark.parametrize("Dk", [32, 64])
@pytest.mark.parametrize("B,H,L", [(1, 1, 129), (3, 2, 196), (1, 2, 224), (130, 2, 200), (64, 2, 140)])
def test_forward(B, H, L, Dk, gates):
    announce(f"fp32 halves forward B{B} H{H} L{L} Dk{Dk} {gates}")
    q, k, v, gf, gb = make_gla_inputs(B, H, L, Dk, 64, seed=L, dtype=torch.float32)
    if gates != "mild":  # in every third sequence one direction's gates leave the form's range, in every fourth the other's
        m, n = ((torch.arange(B * H) % i == 1).reshape(B, H)[:, :, None, None] for i in (3, 4))
        gf, gb = torch.where(m, 60 * gf, gf), torch.where(n, 60 * gb, gb)
        if gates == "positive":  # (one that grows: token by token)
            gf[:, :, :1], gb[:, :, -1:] = torch.where(m, 2.0, gf[:, :, :1]), torch.where(n, 2.0, gb[:, :, -1:])
    t = [x.cuda() for x in (q, k, v, gf, gb)]
    lib = _lib.load()
    most = lib.vig_gla_bidir_fwd_workspace_for(B, H, L, Dk, 64, 0, 0, 1)
    pick = sorted({0, B // 2, B - 1})
    want = oracle_bidir(*(x[pick].cpu() for x in t))
    assert most > 0
    for size in (most, 0):
        o = torch.empty_like(t[2])
        ws = torch.full((size + 512,), 77, dtype=torch.uint8, device="cuda")
        rc = lib.vig_gla_bidir_fwd(*(x.data_ptr() for x in t), o.data_ptr(), ws.data_ptr() if size else None, size, B, H, L, Dk, 64, Dk ** -0.5,
                                   1.0, 0, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == _lib.VIG_OK and (ws[size:] == 77).all()
        assert max_rel(f64(o[pick]), want) <= 1e-5
