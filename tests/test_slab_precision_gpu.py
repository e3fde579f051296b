"""The one-launch forward of many tiles against fp64: no more error than the form it stands for, segments linked by fp32 states."""
import pytest
import torch

import vig_amd
from vig_amd.synthetic import make_gla_inputs

from .util import announce, f64, oracle_bidir

pytestmark = pytest.mark.gpu


# The segments' error, output not yet rounded, is 4.7e-4 to 5.8e-4 of the output's rms at these lengths and gate logits up to 7, and a tenth is
# allowed for the sample; with the decays of the tiles passed taken one by one in fp16 it was 7.3e-4 and 6.9e-4 at logits of 5.
@pytest.mark.parametrize("logit", [0.0, 5.0, 9.0])
@pytest.mark.parametrize("L,Dk", [(288, 32), (512, 32), (288, 64), (416, 64)])
def test_error(L, Dk, logit):
    announce(f"one-launch precision L{L} Dk{Dk} logits around {logit}")
    q, k, v, _, _ = make_gla_inputs(4, 3, L, Dk, 64, seed=L + Dk, dtype=torch.bfloat16)
    gen = torch.Generator().manual_seed(L)
    gf, gb = ((torch.nn.functional.logsigmoid(torch.randn(q.shape, generator=gen) + logit) / 16).bfloat16() for _ in "fb")
    q, k, v, gf, gb = (t.cuda() for t in (q, k, v, gf, gb))
    want = oracle_bidir(q, k, v, gf, gb)
    got = f64(vig_amd.gla_bidir_forward(q, k, v, gf, gb))
    size = (want ** 2).mean()
    rest = ((got - want) ** 2).mean() - ((f64(torch.from_numpy(want).bfloat16()) - want) ** 2).mean()  # without the output's own rounding
    assert rest <= size * 6.4e-4 ** 2
