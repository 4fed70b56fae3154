"""Loader of the native host path (``csrc/torch_calls.cpp``, module ``_torch_calls``).

``calls()`` is the module, bound to the library that ``_capi`` loaded, or None where it was
not built: the operators then run their Python path for every call. Its functions return
None for calls that are not plain eager ones, which the Python path serves as well.
"""
from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import os
import threading
import warnings

import torch

from . import _capi
from ._build import TORCH_CALLS_PATH

__all__ = ["calls"]

# the order of struct Lib in torch_calls.cpp
_ENTRY_POINTS = ("prefixlm_fwd", "prefixlm_bwd", "prefixlm_fwd_q_amax_count", "prefixlm_fwd_workspace_size",
                 "prefixlm_bwd_workspace_size", "prefixlm_bwd_ds_bytes", "prefixlm_bwd_ds_bytes_blocks",
                 "prefixlm_rope", "prefixlm_swiglu_fwd", "prefixlm_swiglu_bwd", "prefixlm_rmsnorm_fwd",
                 "prefixlm_rmsnorm_bwd", "prefixlm_add_rmsnorm", "prefixlm_proj_gemm", "prefixlm_proj_gemm_scaled",
                 "prefixlm_kvcache_workspace_size", "prefixlm_kvcache_fwd", "prefixlm_last_error")

_lock = threading.Lock()
_module = None
_done = False


def _load():
    global _module, _done
    with _lock:
        if _done:
            return
        mod = None
        if os.path.exists(TORCH_CALLS_PATH) and os.path.exists(_capi.lib_path()):
            try:
                loader = importlib.machinery.ExtensionFileLoader("_torch_calls", TORCH_CALLS_PATH)
                spec = importlib.util.spec_from_file_location("_torch_calls", TORCH_CALLS_PATH, loader=loader)
                mod = importlib.util.module_from_spec(spec)
                loader.exec_module(mod)
            except ImportError as e:
                warnings.warn(f"prefixlm: {TORCH_CALLS_PATH} does not load ({e}); rebuild the extension. "
                              "Calls take the slower Python host path.")
                mod = None
        if mod is not None:
            lib = _capi.load()
            caps = [torch.cuda.get_device_properties(i).total_memory // 8 for i in range(torch.cuda.device_count())]
            mod.bind([ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in _ENTRY_POINTS], caps,
                     torch.nn.Parameter)
            mod.set_timer(_capi.active_timer().value)
            _capi.Timer.on_change = mod.set_timer
        _module = mod
        _done = True


def calls():
    """The native module, or None."""
    if not _done:
        _load()
    return _module
