"""The fp32 backward with both directions' key operands in LDS (32 key channels; three tiles and five to seven): lengths around the tiles'
edges, whole sequences and segments, sequences out of the form's range, against the fp64 oracle."""
import pytest
import torch

from oracle import gla_oracle as O
from vig_amd import _lib
from vig_amd.synthetic import make_gla_inputs

from .test_backward_gpu import _check_all
from .test_f32_halves_gpu import _run
from .util import announce, f64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("strong", [False, True])
@pytest.mark.parametrize("L", [64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 257, 450, 1100])
def test_against_oracle(L, strong):
    B, H, Dk = 2, 3, 32
    announce(f"fp32 both directions L{L} strong={strong}")
    q, k, v, gf, gb = make_gla_inputs(B, H, L, Dk, 64, seed=L, dtype=torch.float32)
    if strong:  # every third sequence is flagged, by either direction's gates
        m, n = ((torch.arange(B * H) % 3 == i).reshape(B, H)[:, :, None, None] for i in (1, 2))
        gf, gb = torch.where(m, 60 * gf, gf), torch.where(n, 60 * gb, gb)
    do = torch.randn(v.shape, generator=torch.Generator().manual_seed(L))
    t = [x.cuda() for x in (q, k, v, gf, gb, do)]
    # (the smallest workspace: whole items, no halves)
    got = _run(*t, _lib.load().vig_gla_bidir_bwd_workspace(B, H, L, Dk, 64, 1))
    _check_all(got, O.bidir_gla_backward(*(f64(x) for x in t)), q, tol=1e-5)
