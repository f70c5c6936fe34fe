"""Native call marshalling (csrc/fa_torch.cpp) for the plain case of each entry point.

Each function returns the entry point's result, raises what the library's
status says, or returns None when the call is not the plain case (CPU or
foreign-device tensors, subclasses, conversions or copies needed, mistakes):
the caller's Python path then takes it, with its checks and messages.  The
same where the extension is not built for this torch: every call then goes
through ctypes to the same kernels, after one warning.
"""
from __future__ import annotations

import ctypes
import threading
import warnings

import torch

from . import _lib

_ENTRIES = ("fa_fwd", "fa_decode_workspace_bytes", "fa_paged_decode",
            "fa_paged_prefill_num_splits", "fa_paged_prefill_splitkv_workspace_bytes",
            "fa_paged_prefill_splitkv", "fa_reshape_and_cache")
_lock = threading.Lock()
_module = None
_missing = False  # load() failed: the Python path takes every call


def load():
    """The extension module, bound to the library's entry points; RuntimeError where it is not
    built for this torch."""
    global _module
    if _module is None:
        lib = _lib.load()
        with _lock:
            if _module is None:
                try:
                    from . import _fa_torch
                    built = getattr(_fa_torch, "torch_version", None)
                    if built != torch.__version__:
                        raise ImportError(f"built for torch {built}")
                except ImportError as e:
                    raise RuntimeError(
                        f"_fa_torch is not built for this torch ({e}); run "
                        "`python tilelang-fa-v100_amd/build.py` (or __graft_entry__.build())"
                    ) from e
                _fa_torch.bind(*(ctypes.cast(getattr(lib, n), ctypes.c_void_p).value
                                 for n in _ENTRIES))
                _module = _fa_torch
    return _module


def _extension():
    """load(), or None with one warning."""
    global _missing
    _lib.load()  # the kernels themselves: an error for every call
    try:
        return load()
    except RuntimeError as e:
        with _lock:
            first, _missing = not _missing, True
        if first:
            warnings.warn(f"{e}; calls are marshalled in Python (several us more each)",
                          RuntimeWarning, stacklevel=2)
        return None


def _run(name, what, first, args):
    if _missing or not (isinstance(first, torch.Tensor) and first.is_cuda):
        return None
    module = _module or _extension()
    if module is None:
        return None
    device = torch._C._cuda_getDevice()
    r = getattr(module, name)(*args, device, torch._C._cuda_getCurrentRawStream(device))
    if type(r) is int:
        _lib.check(r, what)
    return r


def dense_forward(q, k, v, scale, causal, window, with_lse):
    """(out, lse or None), or None."""
    if type(window) is not tuple or len(window) != 2:
        return None
    return _run("dense_forward", "fa_fwd", q,
                (q, k, v, scale, bool(causal), window[0], window[1], with_lse))


def decode(q, *args):
    """out, or None."""
    return _run("decode", "fa_paged_decode", q, (q, *args))


def paged_forward(q, k_cache, v_cache, block_table, seq_lens, query_start_loc, prefix_kv_lens,
                  block_size, num_kv_heads, scale, causal, window_q, window_k):
    """(out, lse), or None."""
    return _run("paged_forward", "fa_paged_prefill_splitkv", q,
                (q, k_cache, v_cache, block_table, seq_lens, query_start_loc, prefix_kv_lens,
                 block_size, num_kv_heads, scale, bool(causal), window_q, window_k))


def cache_write(key, *args):
    """0, or None."""
    return _run("cache_write", "fa_reshape_and_cache", key, (key, *args))
