"""Loads csrc/host.cpp's extension (built beside the kernel library) and hands it the C ABI's addresses.

The extension serves the operators' plain calls; see its header comment. It holds no kernels: where it is
missing, or was built for another torch or Python than the running ones (whose C++ types it uses), the
Python path serves every call, with the same results and after one warning.
"""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import sys
import threading
import warnings
from pathlib import Path

from . import _abi

_PATH = Path(__file__).resolve().parent / "_lib" / "w4a8_host.so"

# the members of host.cpp's Abi, in their order
_ENTRY_POINTS = (
    "w4a8_last_error", "w4a8_linear", "w4a8_linear_workspace_bytes_for", "w4a8_gemm", "w4a8_gemm_workspace_bytes",
    "w4a8_rms_norm", "w4a8_moe_padded_capacity", "w4a8_moe_route_gemm1", "w4a8_moe_route_slots",
    "w4a8_moe_route_align", "w4a8_moe_gemm_workspace_bytes", "w4a8_moe_gemm", "w4a8_moe_gemm2_combine_supported",
    "w4a8_moe_gemm2_combine", "w4a8_moe_gemm_quant_workspace_bytes", "w4a8_moe_gemm_quant", "w4a8_moe_combine",
)

_lock = threading.Lock()
_mod = None


class _Absent:
    """In the extension's place: takes no call."""

    linear = rms_norm = moe = staticmethod(lambda *a: None)


def _running() -> str:
    """What the extension must have been built for (build.py's form)."""
    import torch

    return f"torch {torch.__version__}, Python {sys.version_info.major}.{sys.version_info.minor}"


def _extension():
    """The extension module, or ImportError with the reason it cannot be used."""
    want = _running()  # imports torch, whose libraries must be loaded before the extension
    if not _PATH.exists():
        raise ImportError(f"{_PATH} is not built")
    loader = importlib.machinery.ExtensionFileLoader("w4a8_host", str(_PATH))
    mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("w4a8_host", loader))
    loader.exec_module(mod)
    if getattr(mod, "built_for", None) != want:
        raise ImportError(f"{_PATH} is built for {getattr(mod, 'built_for', 'an unknown torch')}, this is {want}")
    return mod


def load():
    """The extension module, loaded and bound once, or its stand-in."""
    global _mod
    if _mod is not None:
        return _mod
    with _lock:
        if _mod is None:
            lib = _abi.load()
            try:
                mod = _extension()
                mod.bind(*(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _ENTRY_POINTS))
            except ImportError as e:
                warnings.warn(f"w4a8 operators take their slower Python host path ({e}); run "
                              f"__graft_entry__.build() or python minisglang-rdna4_amd/build.py", RuntimeWarning,
                              stacklevel=3)
                mod = _Absent
            _mod = mod
    return _mod
