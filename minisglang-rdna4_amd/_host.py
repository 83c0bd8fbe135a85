"""Loads csrc/host.cpp's extension (built beside the kernel library) and hands it the C ABI's addresses.

The extension serves the operators' plain calls; see its header comment. Like the kernel library it has
no fallback: a GPU call without it raises.
"""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import threading
from pathlib import Path

from . import _abi

_PATH = Path(__file__).resolve().parent / "_lib" / "w4a8_host.so"

# the members of host.cpp's Abi, in their order
_ENTRY_POINTS = (
    "w4a8_last_error", "w4a8_linear", "w4a8_linear_workspace_bytes", "w4a8_gemm", "w4a8_gemm_workspace_bytes",
    "w4a8_rms_norm", "w4a8_moe_padded_capacity", "w4a8_moe_route_gemm1", "w4a8_moe_route_slots",
    "w4a8_moe_route_align", "w4a8_moe_gemm_workspace_bytes", "w4a8_moe_gemm", "w4a8_moe_gemm2_combine_supported",
    "w4a8_moe_gemm2_combine", "w4a8_moe_gemm_quant_workspace_bytes", "w4a8_moe_gemm_quant", "w4a8_moe_combine",
)

_lock = threading.Lock()
_mod = None


def load():
    """The extension module, loaded and bound once."""
    global _mod
    if _mod is not None:
        return _mod
    with _lock:
        if _mod is None:
            import torch  # noqa: F401  (its libraries must be loaded before the extension)

            lib = _abi.load()
            if not _PATH.exists():
                raise RuntimeError(f"w4a8_host.so not built ({_PATH}); run __graft_entry__.build() or "
                                   f"python minisglang-rdna4_amd/build.py")
            loader = importlib.machinery.ExtensionFileLoader("w4a8_host", str(_PATH))
            mod = importlib.util.module_from_spec(importlib.util.spec_from_loader("w4a8_host", loader))
            loader.exec_module(mod)
            mod.bind(*(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _ENTRY_POINTS))
            _mod = mod
    return _mod
