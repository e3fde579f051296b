"""The static checks of test_isa_hazards.py on the matrix-core kernels of few rows and images, the LDS-tiled products, and the bf16 backward on rows."""
import re

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


def test_many_tiles_send_no_more_through_memory():
    # whole sequences past 256 tokens, 64 key channels, both directions: q^ of the second direction waits in memory, and little else (seven
    # reloads more: 33 sequences of 275 tokens 14.6 -> 16.7 us)
    asm = _assembly("gla_tiles.hip")
    name, = re.findall(r"^(_ZN3vig15gla_tile_kernelILi4ELb1ELb0ELb0ELb0ELb0ELb1E\w*):", asm, re.M)
    body = re.search(rf"^{name}:.*?^\.Lfunc_end", asm, re.S | re.M).group(0)
    assert body.count("scratch_load") <= 20 and body.count("scratch_store") <= 20


def test_recurrent_backward_of_16_channels_leaves_room_for_six_waves():
    # 512 registers a SIMD, whole eights a wave (with 96: 3072 sequences of 98 tokens 411 -> 456 us)
    asm = _assembly("gla_backward.hip")
    counts = re.findall(r"\.name:\s+_ZN3vig19gla_backward_kernelI\w\wLi16E.*?\.vgpr_count:\s+(\d+)", asm, re.S)
    assert len(counts) == 4 and all(int(n) <= 80 for n in counts), counts
