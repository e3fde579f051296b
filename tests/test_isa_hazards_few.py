"""The static checks of test_isa_hazards.py on the matrix-core kernels of few rows and images, the LDS-tiled products, and the bf16 backward on rows."""
import pytest

from .test_isa_hazards import _assembly, _report, early_reads, reloads_while_staging


@pytest.mark.parametrize("src", ["conv_linear.hip", "blend_swiglu.hip", "gemm.hip"])
def test_no_early_read_of_matrix_results(src):
    asm = _assembly(src)
    assert "v_mfma_" in asm
    hits = early_reads(asm)
    assert hits == [], _report(hits)


def test_no_reload_between_the_directions_on_rows():
    # whole sequences, 64 key channels: two to eight waves, both directions
    found, seen = reloads_while_staging(_assembly("gla_backward_mfma.hip"), r"_ZN3vig24gla_backward_rows_kernelILi4ELi[23478]E")
    assert seen == 10 and found == []
