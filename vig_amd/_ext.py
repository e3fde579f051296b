"""Loader of the PyTorch-ROCm operator library (vig_amd/lib/libvig_torch_ext.so, built from csrc/torch_ext.cpp).

The operators (torch.ops.vig_amd.*) are the same C-ABI entry points as the ctypes binding reaches, with the argument
checks, output allocation and stream lookup done in C++: one dispatcher call instead of a few dozen Python
statements per kernel.  The ctypes binding stays the torch-free way in; VIG_AMD_NO_EXT=1 keeps this package on it.
"""
from __future__ import annotations

import os

_HERE = os.path.dirname(os.path.abspath(__file__))
EXT_PATH = os.path.join(_HERE, "lib", "libvig_torch_ext.so")

CALLS_PATH = os.path.join(_HERE, "lib", "vig_host.so")

_ops = None
_tried = False
_error = None
_calls = None
_calls_tried = False


def load():
    """torch.ops.vig_amd, or None when the operator library is not built, fails to load or is switched off."""
    global _ops, _tried, _error
    if _tried:
        return _ops
    _tried = True
    if os.environ.get("VIG_AMD_NO_EXT") == "1":
        _error = "switched off by VIG_AMD_NO_EXT=1"
        return None
    if not os.path.exists(EXT_PATH):
        _error = f"{EXT_PATH} is not built (python -m vig_amd.build)"
        return None
    try:
        import torch

        torch.ops.load_library(EXT_PATH)
        _ops = torch.ops.vig_amd
    except Exception as e:  # an operator library built against another torch: the ctypes binding still works
        _error = f"{type(e).__name__}: {e}"
        _ops = None
        import warnings

        warnings.warn(f"vig_amd: {EXT_PATH} exists but did not load ({_error}); falling back to the ctypes binding, "
                      "which costs about twice the host time per call. Rebuild it with `python -m vig_amd.build`.",
                      RuntimeWarning, stacklevel=2)
    return _ops


def calls():
    """The op-level calls as a CPython module (vig_amd/lib/vig_host.so, built from csrc/py_calls.cpp), or None when it is not
    built, fails to load or is switched off (VIG_AMD_NO_EXT=1): ops.py then goes through ctypes."""
    global _calls, _calls_tried
    if _calls_tried:
        return _calls
    _calls_tried = True
    if os.environ.get("VIG_AMD_NO_EXT") == "1" or not os.path.exists(CALLS_PATH):
        return None
    try:
        import importlib.machinery
        import importlib.util

        import torch  # noqa: F401  (the module links to torch's libraries)

        loader = importlib.machinery.ExtensionFileLoader("vig_host", CALLS_PATH)
        spec = importlib.util.spec_from_file_location("vig_host", CALLS_PATH, loader=loader)
        mod = importlib.util.module_from_spec(spec)
        loader.exec_module(mod)
        _calls = mod
    except Exception as e:  # built against another torch or Python: the ctypes binding still works
        import warnings

        warnings.warn(f"vig_amd: {CALLS_PATH} exists but did not load ({type(e).__name__}: {e}); falling back to the "
                      "ctypes binding, whose calls take about 20 us of host time. Rebuild it with "
                      "`python -m vig_amd.build`.", RuntimeWarning, stacklevel=2)
    return _calls


def why_not() -> str | None:
    """Why load() returned None (for diagnostics), or None if it did not."""
    load()
    return _error
