"""ctypes binding of ``libqmm.so`` (declarations in ``include/qmm.h``)."""
from __future__ import annotations

import ctypes as C
import os
import sys
import warnings

import torch

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libqmm.so")
CALL_PATH = os.path.join(HERE, "_call.so")

QMM_F32, QMM_BF16, QMM_F16 = 0, 1, 2
QMM_FLAG_W_BF16 = 1
QMM_FLAG_ACT_Q8K = 2
QMM_FLAG_OUT_BF16 = 4
QMM_OP_MATMUL, QMM_OP_RMSNORM, QMM_OP_SWIGLU, QMM_OP_REPACKED = 0, 1, 2, 3
QMM_STATIC_SCRATCH_BYTES = 64 * 1024 * 1024


class GptqConfig(C.Structure):
    _fields_ = [("bits", C.c_int32), ("group_size", C.c_int32), ("desc_act", C.c_int32), ("sym", C.c_int32)]


_i64, _int, _vp = C.c_int64, C.c_int, C.c_void_p

# name -> (restype, argtypes); every symbol include/qmm.h declares
SIGNATURES = {
    "qmm_version": (_int, []),
    "qmm_last_error": (C.c_char_p, []),
    "qmm_block_params": (_int, [_int, C.POINTER(_i64), C.POINTER(_i64)]),
    "qmm_device_info": (_int, [C.POINTER(C.c_int32), C.POINTER(C.c_int32)]),
    "qmm_read_probe": (_int, [_vp, _i64, _vp]),
    "qmm_mfma_probe": (_int, [_vp, _i64, _int, _int, C.POINTER(_i64), _vp]),
    "qmm_dequantize": (_int, [_int, _vp, _i64, _i64, _vp, _int, _vp]),
    "qmm_dequantize_gptq": (_int, [C.POINTER(GptqConfig), _vp, _vp, _vp, _vp, _i64, _i64, _vp, _int, _vp]),
    "qmm_quantize": (_int, [_int, _vp, _i64, _i64, _vp, _vp]),
    "qmm_quantize_gptq": (_int, [C.POINTER(GptqConfig), _vp, _i64, _i64, _vp, _vp, _vp, _vp, _vp]),
    "qmm_matmul_workspace_bytes": (_i64, [_int, _int, _i64, _i64, _i64]),
    "qmm_matmul_workspace_bytes_flags": (_i64, [_int, _int, _i64, _i64, _i64, _int]),
    "qmm_preferred_workspace_bytes": (_i64, [_int, _int, C.POINTER(GptqConfig), _int, _i64, _i64, _i64, _int]),
    "qmm_matmul": (_int, [_int, C.POINTER(GptqConfig), _vp, _int, _i64, _i64, C.POINTER(_vp), _int, _i64, _vp, _vp,
                          _i64, _int, _vp]),
    "qmm_matmul_static": (_int, [_int, C.POINTER(GptqConfig), _vp, _int, _i64, _i64, C.POINTER(_vp), _int, _i64, _vp, _int,
                                 _vp]),
    "qmm_repack_bytes": (_i64, [_int, C.POINTER(GptqConfig), _i64, _i64]),
    "qmm_repack": (_int, [_int, C.POINTER(GptqConfig), C.POINTER(_vp), _int, _i64, _i64, _vp, _i64, _vp]),
    "qmm_repack_check": (_int, [_int, C.POINTER(GptqConfig), _i64, _i64, _vp, _i64, _vp]),
    "qmm_matmul_repacked_workspace_bytes": (_i64, [_int, _int, _i64, _i64, _i64]),
    "qmm_matmul_repacked": (_int, [_int, C.POINTER(GptqConfig), _vp, _int, _i64, _i64, C.POINTER(_vp), _int, _vp, _i64, _i64, _vp,
                                   _vp, _i64, _int, _vp]),
    "qmm_matmul_grouped_workspace_bytes": (_i64, [_int, _int, _i64, _i64, _int, C.POINTER(_i64)]),
    "qmm_matmul_grouped": (_int, [_int, _vp, _int, _i64, _i64, _int, C.POINTER(_vp), C.POINTER(_i64), C.POINTER(_vp), _vp,
                                  _i64, _vp]),
    "qmm_matmul_swiglu_workspace_bytes": (_i64, [_int, _int, _i64, _i64, _i64]),
    "qmm_matmul_swiglu": (_int, [_int, _vp, _int, _i64, _i64, _vp, _vp, _i64, _vp, _vp, _i64, _vp]),
    "qmm_matmul_rmsnorm_workspace_bytes": (_i64, [_int, _int, _i64, _i64, _i64, _int]),
    "qmm_matmul_rmsnorm": (_int, [_int, C.POINTER(GptqConfig), _vp, _int, _vp, C.c_float, _i64, _i64, C.POINTER(_vp), _int, _i64,
                                  _vp, _vp, _i64, _int, _vp]),
    "qmm_block_dots_q4_0": (_int, [_vp, _vp, _i64, _i64, _i64, _vp, _vp]),
}

_lib = None


def load() -> C.CDLL:
    """dlopen the library; a missing build is an error, never a fallback."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is not built; run `python -m mojo_amd.build` (hipcc, gfx950). "
                "There is no fallback path without it.")
        lib = C.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(lib, name)
            fn.restype = res
            fn.argtypes = args
        _lib = lib
    return _lib


_call = None


class _Declines:
    """In place of ``mojo_amd._call`` where that does not load: every function declines every call."""

    def __getattr__(self, name):
        return lambda *args: None


def call_stamp() -> str:
    """What ``_call.so`` is bound to: it reads torch's C++ objects, whose layout another torch (or Python) may change."""
    return f"qmm_call for torch {torch.__version__} {torch.version.git_version} {sys.implementation.cache_tag};"


def call_is_current(path: str) -> bool:
    """Whether the module file at ``path`` was compiled for this torch and Python (its bytes hold their stamp); nothing is loaded."""
    try:
        with open(path, "rb") as f:
            return call_stamp().encode() in f.read()
    except OSError:
        return False


def call():
    """The extension module ``mojo_amd._call`` (``csrc/py_call.cpp``).

    It is only the quicker way to ``libqmm.so``: where it is missing (a Python without its headers), does not
    load or was compiled for another torch, a warning says so once and every call takes the Python code in ``ops.py``, which
    reaches the same kernels through ctypes.  Without ``libqmm.so`` this raises as :func:`load` does."""
    global _call
    if _call is None:
        load()
        try:
            if os.path.exists(CALL_PATH) and not call_is_current(CALL_PATH):
                raise ImportError("it was compiled for another torch or Python")
            from . import _call as native
        except ImportError as e:
            warnings.warn(f"mojo_amd/_call.so is not built or does not load ({e}): calls go through ctypes, some 8 us slower each; "
                          "`python -m mojo_amd.build` builds it", RuntimeWarning, stacklevel=3)
            _call = _Declines()
            return _call
        from .quantization import _BLOCKS, _CODES

        native.setup([(enc, code, *((_BLOCKS[enc].elements_per_block, _BLOCKS[enc].block_size) if enc in _BLOCKS else (0, 0)))
                      for enc, code in _CODES.items()])
        _call = native
    return _call


class QmmError(RuntimeError):
    pass


def check(rc: int, what: str) -> None:
    if rc == 0:
        return
    msg = load().qmm_last_error().decode("utf-8", "replace")
    if rc == -1:
        raise ValueError(f"{what}: {msg}")
    if rc == -2:
        raise NotImplementedError(f"{what}: {msg}")
    raise QmmError(f"{what} failed ({rc}): {msg}")
