"""The C-ABI library loads and exports every symbol include/vig_gla.h declares (no GPU)."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "vig_gla.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(vig_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_expected_entry_points():
    syms = _declared_symbols()
    for s in ("vig_gla_bidir_fwd", "vig_gla_bidir_fwd_workspace", "vig_dirgate_fwd", "vig_locality_gate_fwd"):
        assert s in syms


def test_library_exports_every_declared_symbol():
    from vig_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here (python -m vig_amd.build)")
    lib = _lib.load()
    for s in _declared_symbols():
        assert hasattr(lib, s), f"{s} declared in vig_gla.h but not exported"
        assert s in _lib.SIGNATURES, f"{s} has no ctypes signature"
    assert b"gfx950" in lib.vig_gla_version()


def test_argument_validation_without_gpu():
    """Bad arguments are rejected before anything touches a device."""
    from vig_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    lib = _lib.load()
    rc = lib.vig_gla_bidir_fwd(None, None, None, None, None, None, None, 0, 1, 1, 1, 64, 64, 1.0, 1.0, 0, 0, None)
    assert rc == -22
    one = 1 << 20  # non-null dummy addresses; the call must fail on shape before any launch
    rc = lib.vig_gla_bidir_fwd(one, one, one, one, one, one, None, 0, 1, 1, 8, 48, 64, 1.0, 1.0, 0, 0, None)
    assert rc == -95
    rc = lib.vig_gla_bidir_fwd(one, one, one, one, one, one, None, 0, 0, 1, 8, 64, 64, 1.0, 1.0, 0, 0, None)
    assert rc == -22
    rc = lib.vig_gla_bidir_fwd_exact(one, one, one, one, one, one, None, 0, 1, 1, 8, 64, 64, 1.0, 1.0, 1, 1, None)
    assert rc == -28  # bf16 bidirectional exact path needs workspace
    assert lib.vig_gla_strerror(-28) == b"workspace too small"
    assert lib.vig_dirgate_fwd(one, one, 1, 1, 1, 12, 1.0, 0.0, 0, 0, None) == -95
    # launch geometry is checked before anything is enqueued: B*H beyond int range, row counts beyond int range, and
    # more (sequence, direction) pairs than the long-sequence scan's grid takes
    assert lib.vig_gla_bidir_fwd(one, one, one, one, one, one, one, 1 << 40, 40000, 2, 300, 64, 64, 1.0, 1.0, 1, 1,
                                 None) == -95
    # one direction: 40000 pairs fit the grid, so the call gets as far as the workspace check, which refuses it (no
    # workspace is offered: a call on dummy addresses must never reach a launch)
    assert lib.vig_gla_bidir_fwd(one, one, one, one, None, one, None, 0, 40000, 1, 300, 64, 64, 1.0, 1.0, 1, 1,
                                 None) == -28
    big = 1 << 40
    assert lib.vig_gla_bidir_bwd(one, one, one, one, one, one, one, one, one, one, one, one, big, 70000, 70000, 8, 64,
                                 64, 1.0, 1.0, 1, 1, None) == -22
    assert lib.vig_rmsnorm_bwd(one, one, one, None, one, None, None, 0, 1 << 31, 384, 1e-6, 1, None) == -22
    assert lib.vig_gla_bidir_fwd_workspace_for(128, 6, 196, 64, 64, 1, 1, 1) == 0
    assert lib.vig_gla_bidir_fwd_workspace_for(128, 6, 196, 64, 64, 1, 0, 1) == 128 * 6 * 196 * 64 * 4
    assert lib.vig_gla_bidir_fwd_workspace_for(2, 3, 197, 64, 64, 1, 0, 0) == 0


def test_ops_refuse_cpu_tensors():
    import torch

    import vig_amd
    from vig_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    q = torch.zeros(1, 1, 4, 64)
    with pytest.raises(_lib.VigGlaError):
        vig_amd.gla_bidir_forward(q, q, q, q, q)


def test_reference_signatures():
    """Positional order and defaults of the mirrored ops (chunk_fuse.py:554-596, recurrent_fuse.py:659-669)."""
    import inspect

    import vig_amd

    p = list(inspect.signature(vig_amd.fused_chunk_gla).parameters)
    assert p == ["q", "k", "v", "g", "scale", "initial_state", "output_final_state"]
    p = list(inspect.signature(vig_amd.batch_bid_fused_chunk_gla).parameters)
    assert p == ["q", "k", "v", "g", "scale", "initial_state", "output_final_state"]
    sig = inspect.signature(vig_amd.bid_fused_recurrent_gla)
    assert list(sig.parameters) == ["q", "k", "v", "gk", "gv", "scale", "initial_state", "output_final_state", "causal"]
    assert sig.parameters["scale"].default == -1 and sig.parameters["causal"].default is True


def test_token_rows_past_two_to_the_31():
    """Elementwise passes over token rows take as many as 32 bits number (16 channels of them fit the card)."""
    import torch

    from vig_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    if torch.cuda.is_available():
        pytest.skip("pointers to nothing: only where no launch can follow")
    lib, p, nan = _lib.load(), 4096, float("nan")
    refused = (_lib.VIG_EINVAL, _lib.VIG_ENOTSUP)
    for B, L in ((2, 1 << 30), (60000, 70000)):
        assert lib.vig_dirgate_fwd(p, p, B, L, 1, 8, 1.0, nan, 1, 1, None) not in refused
        assert lib.vig_dirgate_bwd(p, p, p, B, L, 1, 8, 1.0, nan, 1, 1, None) not in refused
        assert lib.vig_split_heads_fwd(p, p, p, p, B, L, 1, 8, 8, 0, 1, None) not in refused
    assert lib.vig_dirgate_fwd(p, p, 65535, 70000, 1, 8, 1.0, nan, 1, 1, None) in refused


def test_stem_norm_rows_a_walk_can_step_past():
    """The backward walks rows in steps of up to 16384 (8 to 128 channels) and counts them as ints: rows that a step could carry past 2^31 - 1 are refused."""
    import torch

    from vig_amd import _lib

    if torch.cuda.is_available() or not os.path.exists(_lib.LIB_PATH):
        pytest.skip("pointers to nothing: only where no launch can follow")
    lib, p, last = _lib.load(), 4096, 2 ** 31 - 1 - 512 * (512 // 16)
    fwd = lambda rows, C: lib.vig_stem_norm_fwd(p, None, p, p, p, rows, C, 1e-5, 1, 1, 1, None)  # noqa: E731
    bwd = lambda rows, C: lib.vig_stem_norm_bwd(p, None, p, p, p, p, p, p, 2 ** 40, rows, C, 1e-5, 1, 1, 1, None)  # noqa: E731
    for C in (8, 128, 1024):
        for rows in (last + 1, 2 ** 31 - 8192, 2 ** 31 - 1, 2 ** 31):
            assert fwd(rows, C) == bwd(rows, C) == _lib.VIG_ENOTSUP, (rows, C)
        assert fwd(last, C) not in (_lib.VIG_ENOTSUP, _lib.VIG_EINVAL) and bwd(last, C) not in (_lib.VIG_ENOTSUP, _lib.VIG_EINVAL)  # (no device here)


def test_columns_of_the_norm_convolution_and_product():
    """Its column tiles are 128 wide: the widths it takes, and the ones the header names."""
    from vig_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    takes, p = _lib.load().vig_norm_dwconv3x3_linear_preferred, 4096
    for C in (192, 384):
        assert [N for N in range(8, 641, 8) if takes(1, 4, 8, C, N)] == list(range(128, 641, 128))
        assert _lib.load().vig_norm_dwconv3x3_linear_fwd(p, None, p, p, None, p, None, None, 2 * p, 3 * p, 1, 4, 8, C, 192, 1e-6, 1, None) == _lib.VIG_ENOTSUP
    text = " ".join(open(os.path.join(ROOT, "include", "vig_gla.h")).read().split())
    assert re.search(r"N % (\d+) == 0 and few images \(vig_norm_dwconv3x3_linear_preferred\)", text).group(1) == "128"
