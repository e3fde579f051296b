"""The static check of test_isa_hazards.py over the fp32 (op and products), weight-gradient and linear-layer kernels."""
import pytest

from .test_isa_hazards import test_no_early_read_of_matrix_results as check


@pytest.mark.parametrize("src", ["gla_f32.hip", "gla_backward_f32.hip", "wgrad.hip", "gemm.hip", "gemm_f32.hip"])
def test_no_early_read(src):
    check(src)
