"""ctypes binding of libttfa.so (the C ABI declared in include/ttfa.h).

The library is loaded on first use.  If it is missing, every call raises
``LibraryNotBuilt``: there is no fallback implementation.
"""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import threading
import warnings
from pathlib import Path

import torch

_PKG = Path(__file__).resolve().parent
LIB_PATH = _PKG / "libttfa.so"
NATIVE_PATH = _PKG / "_ttfa_torch.so"

TTFA_BF16 = 0
TTFA_F32 = 1
ABI_VERSION = 7

# Negative status codes of include/ttfa.h.
E_NULL, E_HEAD_DIM, E_GROUP, E_SEQ, E_ALIGN, E_DTYPE, E_SCALE, E_EPS, E_QROWS, E_SCRATCH = (
    -1, -2, -3, -4, -5, -6, -7, -8, -9, -10)
BWD_STATIC_MAX_ROWS = 1 << 20  # TTFA_BWD_STATIC_MAX_ROWS
EXPORTED = ("ttfa_abi_version", "ttfa_strerror", "ttfa_fwd", "ttfa_bwd", "ttfa_bwd_dq",
            "ttfa_bwd_dkdv", "ttfa_varlen_fwd", "ttfa_varlen_bwd", "ttfa_decode_workspace_bytes",
            "ttfa_decode_fwd", "ttfa_qk_prologue_fwd",
            "ttfa_qk_prologue_workspace_bytes", "ttfa_qk_prologue_bwd", "ttfa_bwd_static",
            "ttfa_d128_wide", "ttfa_qk_prologue_fwd_tables", "ttfa_qk_prologue_bwd_tables",
            "ttfa_bwd_workspace_bytes", "ttfa_bwd_ws")


class LibraryNotBuilt(RuntimeError):
    pass


class TTFAError(RuntimeError):
    """A nonzero status from libttfa.so (``code`` < 0: argument error, > 0: hipError_t)."""

    def __init__(self, code: int, msg: str):
        super().__init__(f"{msg} (ttfa status {code})")
        self.code = code


_TENSOR_TYPES = (torch.Tensor, torch.nn.Parameter)
_lock = threading.Lock()
_lib = None

_vp, _i, _f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
_SIGS = {
    "ttfa_abi_version": ([], _i),
    "ttfa_strerror": ([_i], ctypes.c_char_p),
    "ttfa_fwd": ([_vp] * 5 + [_i] * 6 + [_f, _vp], _i),
    "ttfa_bwd": ([_vp] * 10 + [_i] * 6 + [_f, _vp], _i),
    "ttfa_bwd_workspace_bytes": ([_i] * 6, ctypes.c_longlong),
    "ttfa_bwd_ws": ([_vp] * 10 + [_i] * 6 + [_f, _vp], _i),
    "ttfa_bwd_dq": ([_vp] * 8 + [_i] * 6 + [_f, _vp], _i),
    "ttfa_bwd_dkdv": ([_vp] * 8 + [_i] * 6 + [_f, _vp], _i),
    "ttfa_varlen_fwd": ([_vp] * 6 + [_i] * 7 + [_f, _vp], _i),
    "ttfa_varlen_bwd": ([_vp] * 11 + [_i] * 7 + [_f, _vp], _i),
    "ttfa_decode_workspace_bytes": ([_i] * 6, ctypes.c_longlong),
    "ttfa_decode_fwd": ([_vp] * 7 + [_i] * 7 + [_f, _vp], _i),
    "ttfa_qk_prologue_fwd": ([_vp] * 12 + [_i] * 5 + [_f, _vp], _i),
    "ttfa_qk_prologue_workspace_bytes": ([_i] * 5, ctypes.c_longlong),
    "ttfa_qk_prologue_bwd": ([_vp] * 17 + [_i] * 5 + [_vp], _i),
    "ttfa_qk_prologue_fwd_tables": ([_vp] * 7 + [_i] + [_vp] * 5 + [_i] * 5 + [_f, _vp], _i),
    "ttfa_qk_prologue_bwd_tables": ([_vp] * 9 + [_i] + [_vp] * 8 + [_i] * 5 + [_vp], _i),
    "ttfa_bwd_static": ([_vp] * 9 + [_i] * 6 + [_f, _vp], _i),
    "ttfa_d128_wide": ([_i] * 3 + [ctypes.POINTER(_i)] * 2, _i),
}


def d128_wide(B: int, Hq: int, T: int) -> tuple[bool, bool]:
    """(forward, dQ pass) of a bf16 D = 128 shape run the 256-row kernels (no HIP call)."""
    f, d = _i(), _i()
    check(load().ttfa_d128_wide(B, Hq, T, ctypes.byref(f), ctypes.byref(d)))
    return bool(f.value), bool(d.value)


def load() -> ctypes.CDLL:
    """Load (once) and return the library, with argument types declared."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not LIB_PATH.exists():
                raise LibraryNotBuilt(
                    f"{LIB_PATH} is missing: build it with `python -m tinytrain_amd.build` "
                    "(the HIP library is the only implementation of these ops)")
            lib = ctypes.CDLL(str(LIB_PATH))
            for name, (argtypes, restype) in _SIGS.items():
                fn = getattr(lib, name)
                fn.argtypes = argtypes
                fn.restype = restype
            ver = lib.ttfa_abi_version()
            if ver != ABI_VERSION:
                raise LibraryNotBuilt(f"{LIB_PATH} has ABI {ver}, expected {ABI_VERSION}; rebuild it")
            _lib = lib
    return _lib


def plain_cuda(t) -> bool:
    """A real GPU tensor (not a subclass such as a fake tensor): worth asking native()."""
    return type(t) in _TENSOR_TYPES and t.is_cuda


class _OpsOnly:
    """Stands in for the extension where it is missing or does not load: hands every call on
    to the custom ops."""

    @staticmethod
    def _pass(*_):
        return None

    flash_attn = flash_attn_varlen = flash_attn_decode = qk_norm_rope = _pass


_native = None


def _load_native():
    name = f"{__package__}._ttfa_torch"
    loader = importlib.machinery.ExtensionFileLoader(name, str(NATIVE_PATH))
    spec = importlib.util.spec_from_file_location(name, NATIVE_PATH, loader=loader)
    try:
        mod = importlib.util.module_from_spec(spec)
        loader.exec_module(mod)
        return mod
    except (ImportError, OSError) as e:
        warnings.warn(f"{NATIVE_PATH} does not load ({e}); the custom ops take every call, at "
                      "about 0.1 ms more host time each. Build it for this torch with "
                      "`python -m tinytrain_amd.build`.", RuntimeWarning, stacklevel=4)
        return _OpsOnly


def native():
    """Load (once) and return the extension of the native eager path (csrc/torch_native.cpp).
    It calls libttfa.so, whose ABI version is checked first; unlike that library it is built
    against one torch, and the ops run without it."""
    global _native
    if _native is None:
        load()
        with _lock:
            if _native is None:
                _native = _load_native()
    return _native


def strerror(code: int) -> str:
    return load().ttfa_strerror(code).decode()


def check(code: int) -> None:
    if code != 0:
        raise TTFAError(code, strerror(code))
