"""ctypes binding of libgdn_amd.so (the C ABI declared in include/gdn_amd.h).

The library is built in-tree (``make -C gated-delta-network_amd/csrc`` or
``__graft_entry__.build()``).  There is no fallback: if the library is missing
or does not export a symbol, loading raises, so no caller can silently run
anything but the HIP kernels.
"""

from __future__ import annotations

import ctypes
import importlib.machinery
import os
import warnings

LIB_NAME = "libgdn_amd.so"
LIB_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), LIB_NAME)

GDN_OK = 0
GDN_ERR_INVALID = -1
GDN_ERR_LAUNCH = -2
GDN_ERR_WORKSPACE = -3
PREFILL_SCRATCH_BYTES = 64 << 20  # GDN_PREFILL_SCRATCH_BYTES
ABI_VERSION = 4

_P = ctypes.c_void_p
_I = ctypes.c_int
_F = ctypes.c_float
_SZ = ctypes.c_size_t

# name -> (restype, argtypes); mirrors include/gdn_amd.h one to one.
SIGNATURES = {
    "gdn_abi_version": (_I, []),
    "gdn_last_error": (ctypes.c_char_p, []),
    "gdn_decode_fwd": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _F, _P, _P, _I, _P]),
    "gdn_decode_fwd_variant": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _F, _P, _P, _I, _P, _I]),
    "gdn_decode_multi_fwd": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _F, _P, _P, _I, _I, _P, _I]),
    "gdn_decode_fwd_heads": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _F, _P, _P, _I, _I, _I, _I,
                                  _P, _I]),
    "gdn_prefill_workspace_bytes": (_SZ, [_I, _I]),
    "gdn_prefill_workspace_bytes_heads": (_SZ, [_I, _I, _I, _I]),
    "gdn_prefill_fwd": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _F, _P, _P, _P,
                             _SZ, _P]),
    "gdn_prefill_fwd_variant": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _F, _P, _P,
                                     _P, _SZ, _P, _I]),
    "gdn_prefill_fwd_tuned": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _F, _P, _P,
                                   _P, _SZ, _P, _I, _I, _I]),
    "gdn_prefill_fwd_heads": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _I, _I, _F,
                                   _P, _P, _P, _SZ, _P, _I, _I, _I]),
    "gdn_prefill_fwd_noalloc": (_I, [_P, _P, _P, _P, _P, _P, _P, _P, _P, _I, _I, _I, _F, _P, _P,
                                     _P]),
    "gdn_prefill_status_offset": (ctypes.c_longlong, [_I, _I, _I, _I]),
    "gdn_prefill_status": (_I, [_P, _I, _I, _I, _I, _P, _P]),
    "gdn_stream_copy": (_I, [_P, _P, _SZ, _P]),
}


class GdnError(RuntimeError):
    """A launch or runtime failure reported by the HIP library."""


class GdnWorkspaceError(GdnError):
    """The prefill workspace was missing or too small."""


_lib = None


def load(path: str = LIB_PATH) -> ctypes.CDLL:
    """Load (once) and return the HIP library with every prototype set."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(path):
        raise RuntimeError(
            f"{path} is not built; build it with `make -C gated-delta-network_amd/csrc` "
            "or `python -c 'import __graft_entry__ as g; g.build()'`")
    lib = ctypes.CDLL(path)
    for name, (res, args) in SIGNATURES.items():
        fn = getattr(lib, name)  # AttributeError if the symbol is missing
        fn.restype = res
        fn.argtypes = args
    got = lib.gdn_abi_version()
    if got != ABI_VERSION:
        raise RuntimeError(f"{path}: ABI version {got}, expected {ABI_VERSION}")
    _lib = lib
    return lib


_native = None
_native_tried = False


def _native_file() -> str | None:
    """The built extension beside this file, or None."""
    here = os.path.dirname(LIB_PATH)
    files = [os.path.join(here, "_native" + s) for s in importlib.machinery.EXTENSION_SUFFIXES]
    return next((f for f in files if os.path.exists(f)), None)


def native():
    """The native entry of ordinary calls (csrc/gdn_torch.cpp), bound to the
    loaded library, or None where the extension is not built (a tree that holds
    the library alone): the Python path then makes the same C ABI calls.  One
    that is there but does not load, or was built against another torch (whose
    tensors it would misread), is not used either, with a warning."""
    global _native, _native_tried
    if not _native_tried:
        import torch  # (the library alone needs none)
        lib = load()
        module = None
        try:
            from . import _native as module
        except ImportError as e:
            if _native_file() is not None:
                warnings.warn(f"{_native_file()} does not load ({e}): calls take the Python path",
                              RuntimeWarning, stacklevel=2)
        if module is not None:
            built = getattr(module, "torch_version", None)
            if built != torch.__version__:
                warnings.warn(f"gdn_amd._native was built against torch {built}, this is "
                              f"{torch.__version__}: calls take the Python path (rebuild with "
                              "`make -C gated-delta-network_amd/csrc -B native`)",
                              RuntimeWarning, stacklevel=2)
                module = None
        if module is not None:
            module.bind(*(ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in (
                "gdn_decode_fwd", "gdn_decode_multi_fwd", "gdn_decode_fwd_heads", "gdn_prefill_fwd",
                "gdn_prefill_fwd_heads", "gdn_prefill_workspace_bytes_heads")))
        _native, _native_tried = module, True
    return _native


def last_error() -> str:
    return load().gdn_last_error().decode(errors="replace")


def check(rc: int, what: str) -> None:
    """Turn a GDN_* status into the matching Python exception."""
    if rc == GDN_OK:
        return
    msg = last_error() or what
    if rc == GDN_ERR_INVALID:
        raise ValueError(msg)
    if rc == GDN_ERR_WORKSPACE:
        raise GdnWorkspaceError(msg)
    raise GdnError(f"{msg} (status {rc})")
