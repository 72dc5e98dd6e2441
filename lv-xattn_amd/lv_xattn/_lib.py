"""ctypes binding of liblvx.so (the gfx950 kernels behind a C ABI, include/lvx.h).

There is no fallback: if the library is missing or a call is rejected the host
code raises.  PyTorch is used only to own device memory and the stream.
"""
from __future__ import annotations

import ctypes as C
import os
from typing import Optional

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("LVX_LIB") or os.path.join(_HERE, "liblvx.so")

VERSION = 104           # of the library (include/lvx.h) this package is written against
LVX_BF16 = 1
LVX_SPLITS_ROUNDS = 12      # in kv_splits, the bit where the number of rounds begins (include/lvx.h)
LVX_BWD_ROUNDS = 12         # likewise in dkv_accumulate
LVX_F16 = 2
LVX_ERR_SHAPE = -3


class LvxError(RuntimeError):
    pass


class AttnShape(C.Structure):
    _fields_ = [
        ("B", C.c_int32), ("Hq", C.c_int32), ("Hkv", C.c_int32), ("D", C.c_int32),
        ("Lq", C.c_int32), ("Lkv", C.c_int32), ("dtype", C.c_int32), ("scale", C.c_float),
        ("kv_len", C.c_void_p), ("kv_start", C.c_void_p), ("kv_end", C.c_void_p),
        ("bias", C.c_void_p), ("bias_stride_b", C.c_int64), ("bias_stride_h", C.c_int64), ("bias_stride_r", C.c_int64),
    ]


class Tensor4(C.Structure):
    _fields_ = [("ptr", C.c_void_p), ("stride_b", C.c_int64), ("stride_h", C.c_int64), ("stride_s", C.c_int64)]


# every symbol include/lvx.h declares: name -> (restype, argtypes)
_P = C.c_void_p
_SHAPE = C.POINTER(AttnShape)
_T = C.POINTER(Tensor4)
SYMBOLS = {
    "lvx_version": (C.c_int, []),
    "lvx_strerror": (C.c_char_p, [C.c_int]),
    "lvx_max_rounds": (C.c_int, []),
    "lvx_fwd_workspace_bytes": (C.c_size_t, [_SHAPE, C.c_int32, C.c_int32]),
    "lvx_fwd_auto_splits": (C.c_int, [_SHAPE, C.c_int32]),
    "lvx_fwd": (C.c_int, [_SHAPE, _T, _T, _T, _T, _P, C.c_int32, C.c_int32, C.c_int32, _P, C.c_size_t, _P]),
    "lvx_fwd_acc": (C.c_int, [_SHAPE, _T, _T, _T, _T, _P, _T, _P, C.c_int32, C.c_int32, C.c_int32, _P, C.c_size_t, _P]),
    "lvx_fwd_noalloc": (C.c_int, [_SHAPE, _T, _T, _T, _T, _P, C.c_int32, C.c_int32, C.c_int32, _P]),
    "lvx_noalloc_scratch_bytes": (C.c_size_t, []),
    "lvx_merge": (C.c_int, [_SHAPE, _T, _P, _T, _P, C.c_int32, C.c_int32, _P]),
    "lvx_bias_hull": (C.c_int, [_SHAPE, _P, _P, _P]),
    "lvx_bias_is_interval": (C.c_int, [_SHAPE, _P, _P, _P, _P]),
    "lvx_mask_intervals": (C.c_int, [_P, C.c_int32, C.c_int64, C.c_int64, C.c_int32, C.c_int32, C.c_int32, _P, _P, _P]),
    "lvx_bwd_preprocess": (C.c_int, [_SHAPE, _T, _T, _P, C.c_int32, C.c_int32, _P]),
    "lvx_bwd": (C.c_int, [_SHAPE, _T, _T, _T, _T, _P, _P, _T, _T, _T, C.c_int32, C.c_int32, C.c_int32,
                          _P, C.c_size_t, _P]),
    "lvx_bwd_from_o": (C.c_int, [_SHAPE, _T, _T, _T, _T, _T, _P, _T, _T, _T, C.c_int32, C.c_int32, C.c_int32,
                                 _P, C.c_size_t, _P]),
    "lvx_bwd_workspace_bytes": (C.c_size_t, [_SHAPE, C.c_int32]),
    "lvx_bwd_acc_workspace_bytes": (C.c_size_t, [_SHAPE, C.c_int32]),
    "lvx_cast_f32": (C.c_int, [_P, _T, C.c_int32, C.c_int32, C.c_int32, C.c_int32, C.c_int32, _P]),
    "lvx_kv_proj": (C.c_int, [_P, C.c_int64, _P, _P, C.c_int64, C.c_int32, _P, _P, C.c_int64,
                              C.c_int32, C.c_int32, C.c_int32, C.c_int32, _P]),
    "lvx_kv_proj_norm": (C.c_int, [_P, C.c_int64, _P, _P, C.c_int64, C.c_int32, _P, _P, C.c_int64,
                                   C.c_int32, C.c_int32, C.c_int32, _P, C.c_float, _P, _P, C.c_int32, _P]),
    "lvx_k_norm_bwd": (C.c_int, [_P, C.c_int64, _P, C.c_int64, _P, _P, _P, C.c_int64, _P,
                                 C.c_int32, C.c_int32, C.c_int32, _P]),
    "lvx_dx_vis": (C.c_int, [_P, _P, C.c_int64, _P, _P, C.c_int64, C.c_int32, _P, C.c_int64,
                             C.c_int32, C.c_int32, C.c_int32, C.c_int32, _P]),
    "lvx_dw_kv": (C.c_int, [_P, C.c_int64, _P, _P, C.c_int64, _P, _P, C.c_int64, C.c_int32,
                            C.c_int32, C.c_int32, C.c_int32, C.c_int32, _P]),
}

_lib: Optional[C.CDLL] = None


def load() -> C.CDLL:
    """dlopen liblvx.so and type every entry point.  Raises if it is absent or of another version."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise LvxError(
            f"{LIB_PATH} is missing: the HIP kernels are not built. "
            "Run `python lv-xattn_amd/build.py` (needs hipcc); there is no CPU fallback.")
    lib = C.CDLL(LIB_PATH)
    if lib.lvx_version() != VERSION:
        raise LvxError(f"{LIB_PATH} is version {lib.lvx_version()} of the library, this package needs {VERSION}")
    for name, (res, args) in SYMBOLS.items():
        try:
            fn = getattr(lib, name)
        except AttributeError:
            raise LvxError(f"{LIB_PATH} has no {name}: an older build than this package, which needs it") from None
        fn.restype = res
        fn.argtypes = args
    _lib = lib
    return lib


_host = _host_lib = None       # the module, and the library whose functions it calls


def host():
    """The native side of the operators (_lvx_host.so, built with the library), calling the functions of the
    library that load() gives.  Raises if it is absent."""
    global _host, _host_lib
    lib = _lib or load()
    if _host_lib is not lib:
        try:
            from . import _lvx_host
        except ImportError as e:
            raise LvxError("_lvx_host.so is missing or does not load: run `python lv-xattn_amd/build.py`") from e
        _lvx_host.bind({name: C.cast(getattr(lib, name), C.c_void_p).value for name in SYMBOLS})
        _host, _host_lib = _lvx_host, lib
    return _host


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = load().lvx_strerror(rc).decode()
        raise LvxError(f"{what} failed: {msg} (code {rc})")


def stream_ptr() -> int:
    return host().stream_of(-1)         # of the current device


def t4(t: torch.Tensor) -> Tensor4:
    """[B, H, S, D] tensor (any strides, unit last stride) -> lvx_tensor."""
    if t.dim() != 4 or t.stride(3) != 1:
        raise LvxError(f"expected a 4-d tensor with unit last stride, got shape {tuple(t.shape)} "
                       f"strides {t.stride()}")
    return Tensor4(t.data_ptr(), t.stride(0), t.stride(1), t.stride(2))


def ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()
