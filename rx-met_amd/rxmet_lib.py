"""ctypes binding of ``librxmet.so`` (the MI355X C ABI declared in ``include/*.h``).

The library is the only compute path of this package: if it is missing, every entry
point raises instead of falling back to anything else.  Calls pass raw device pointers
(``tensor.data_ptr()``) and PyTorch's current HIP stream, so kernels are ordered with
the caller's other work exactly like aten ops.
"""
from __future__ import annotations

import ctypes
import os
import warnings
from pathlib import Path
from typing import Optional

_PKG = Path(__file__).resolve().parent
LIB_PATH = Path(os.environ.get("RXMET_LIB", _PKG / "librxmet.so"))

_lib: Optional[ctypes.CDLL] = None
_torch_ext = None

c_i64 = ctypes.c_int64
c_int = ctypes.c_int
c_ptr = ctypes.c_void_p
c_float = ctypes.c_float



class QdqLayout(ctypes.Structure):
    """rxmet_qdq_layout: [outer, C0, mid, C1, inner], encoding c0 * C1 + c1."""
    _fields_ = [("outer", c_i64), ("C0", c_i64), ("mid", c_i64), ("C1", c_i64), ("inner", c_i64)]


class QdqNumerics(ctypes.Structure):
    """rxmet_qdq_numerics: io / internal element types, zero_point_shift, 0-dim scale."""
    _fields_ = [("io_dtype", ctypes.c_int32), ("internal_dtype", ctypes.c_int32),
                ("zero_point_shift", ctypes.c_double), ("scalar_scale", ctypes.c_int32),
                ("reserved", ctypes.c_int32)]


class QdqMinMaxEnc(ctypes.Structure):
    """rxmet_qdq_minmax_enc: learnable min / max encodings derived inside the kernels."""
    _fields_ = [("min", c_ptr), ("max", c_ptr), ("symmetric", ctypes.c_int32),
                ("sym_offset", ctypes.c_float), ("min_scale", ctypes.c_float),
                ("reserved", ctypes.c_int32)]


class BlockJob(ctypes.Structure):
    """rxmet_block_job (include/rxmet_layout.h): one tensor widened or narrowed."""
    _fields_ = [("src", c_ptr), ("dst", c_ptr), ("outer", c_i64), ("rows_src", ctypes.c_int32),
                ("rows_dst", ctypes.c_int32), ("groups", ctypes.c_int32),
                ("cols_src", ctypes.c_int32), ("cols_dst", ctypes.c_int32),
                ("reserved", ctypes.c_int32)]


BLOCK_JOBS = 16  # RXMET_BLOCK_JOBS

_LAY = ctypes.POINTER(QdqLayout)
_MME = ctypes.POINTER(QdqMinMaxEnc)
_NUM = ctypes.POINTER(QdqNumerics)

# name -> (restype, argtypes); mirrors include/rxmet_qdq.h and include/rxmet_gru.h
_SIGNATURES = {
    "rxmet_last_error": (ctypes.c_char_p, []),
    "rxmet_abi_version": (c_int, []),
    "rxmet_qdq_workspace_bytes": (c_i64, [c_i64, c_i64, c_i64]),
    "rxmet_qdq_minmax": (c_int, [c_ptr, c_i64, c_i64, c_i64, c_ptr, c_ptr, c_ptr, c_ptr]),
    "rxmet_qdq_forward": (c_int, [c_ptr, c_ptr, c_i64, c_i64, c_i64, c_ptr, c_ptr, c_i64, c_i64,
                                  c_int, c_ptr]),
    "rxmet_qdq_backward": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, c_i64, c_i64, c_i64, c_ptr,
                                   c_ptr, c_i64, c_i64, c_int, c_ptr, c_ptr]),
    "rxmet_qdq_backward_noalloc": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, c_i64, c_i64, c_i64,
                                           c_ptr, c_ptr, c_i64, c_i64, c_int, c_ptr]),
    "rxmet_quantize_forward": (c_int, [c_ptr, c_ptr, c_i64, c_i64, c_i64, c_ptr, c_ptr, c_i64,
                                       c_i64, c_ptr]),
    "rxmet_quantize_backward": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, c_i64, c_i64, c_i64,
                                        c_ptr, c_ptr, c_i64, c_i64, c_ptr, c_ptr]),
    "rxmet_dequantize_forward": (c_int, [c_ptr, c_ptr, c_i64, c_i64, c_i64, c_ptr, c_ptr, c_ptr]),
    "rxmet_dequantize_backward": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, c_i64, c_i64, c_i64,
                                          c_ptr, c_ptr, c_ptr, c_ptr]),
    "rxmet_qdq_workspace_bytes_ex": (c_i64, [_LAY, ctypes.c_int32]),
    "rxmet_qdq_minmax_ex": (c_int, [c_ptr, ctypes.c_int32, _LAY, c_ptr, c_ptr, c_ptr, c_ptr]),
    "rxmet_qdq_forward_ex": (c_int, [c_ptr, c_ptr, _LAY, _NUM, c_ptr, c_ptr, c_i64, c_i64, c_int,
                                     c_ptr]),
    "rxmet_qdq_backward_ex": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, _LAY, _NUM, c_ptr, c_ptr,
                                      c_i64, c_i64, c_int, c_ptr, c_ptr]),
    "rxmet_qdq_forward_minmax": (c_int, [c_ptr, c_ptr, _LAY, _NUM, _MME, c_i64, c_i64, c_ptr]),
    "rxmet_qdq_backward_minmax": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, _LAY, _NUM, _MME,
                                          c_i64, c_i64, c_ptr, c_ptr]),
    "rxmet_quantize_forward_ex": (c_int, [c_ptr, c_ptr, _LAY, _NUM, c_ptr, c_ptr, c_i64, c_i64,
                                          c_ptr]),
    "rxmet_quantize_backward_ex": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, _LAY, _NUM, c_ptr,
                                           c_ptr, c_i64, c_i64, c_ptr, c_ptr]),
    "rxmet_dequantize_forward_ex": (c_int, [c_ptr, c_ptr, _LAY, _NUM, c_ptr, c_ptr, c_ptr]),
    "rxmet_dequantize_backward_ex": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_ptr, _LAY, _NUM, c_ptr,
                                             c_ptr, c_ptr, c_ptr]),
    "rxmet_selftest_mfma": (c_int, [c_int, c_ptr, c_ptr, c_ptr, c_ptr]),
    "rxmet_qdq_encoding_forward": (c_int, [c_ptr, c_ptr, c_i64, c_i64, c_i64, ctypes.c_int32,
                                           ctypes.c_float, ctypes.c_float, c_ptr, c_ptr, c_ptr]),
    "rxmet_qdq_encoding_backward": (c_int, [c_ptr, c_ptr, c_ptr, c_ptr, c_i64, c_i64, c_i64,
                                            ctypes.c_int32, ctypes.c_float, c_ptr, c_ptr, c_ptr]),
    "rxmet_block_copy": (c_int, [ctypes.c_int32, ctypes.POINTER(BlockJob), c_ptr]),
    "rxmet_prof_enable": (c_int, [ctypes.c_int32]),
    "rxmet_prof_filter": (c_int, [ctypes.c_char_p]),
    "rxmet_prof_reset": (c_int, []),
    "rxmet_prof_query": (c_int, [ctypes.c_char_p, ctypes.POINTER(ctypes.c_double),
                                 ctypes.POINTER(c_i64)]),
    "rxmet_prof_names": (c_i64, [ctypes.c_char_p, c_i64]),
}



def exported() -> tuple:
    """Names of every typed entry point (tests check the library exports them all)."""
    return tuple(_SIGNATURES)


class RxmetError(RuntimeError):
    """Raised when a C-ABI call reports a failure (argument or HIP error)."""


def load() -> ctypes.CDLL:
    """Load and type the library once; raise if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not LIB_PATH.exists():
        raise RxmetError(
            f"{LIB_PATH} is missing: build it with `python rx-met_amd/build.py` "
            "(the MI355X kernels have no fallback)")
    lib = ctypes.CDLL(str(LIB_PATH))
    for name, (res, args) in _SIGNATURES.items():
        try:
            fn = getattr(lib, name)
        except AttributeError as e:
            raise RxmetError(f"{LIB_PATH} does not export {name}") from e
        fn.restype = res
        fn.argtypes = args
    _lib = lib
    return lib


def torch_ext():
    """The autograd nodes in C++ (module ``rxmet_torch``, built by build.py), bound to the entry
    points of the loaded library; None, with one warning, where the module cannot be imported (the
    Python functions over the same kernels serve then)."""
    global _torch_ext
    if _torch_ext is not None:
        return _torch_ext or None
    lib = load()
    import torch  # noqa: F401  (the module's symbols come from PyTorch's libraries)

    try:
        import rxmet_torch
    except ImportError as e:
        _torch_ext = False
        warnings.warn(f"the module rxmet_torch cannot be imported ({e}); learnable quantizers run "
                      "through Python autograd functions, which take the host longer per call. "
                      "`python rx-met_amd/build.py` builds it", stacklevel=2)
        return None
    rxmet_torch.bind(*(ctypes.cast(getattr(lib, n), c_ptr).value for n in (
        "rxmet_qdq_forward_minmax", "rxmet_qdq_backward_minmax", "rxmet_qdq_workspace_bytes_ex",
        "rxmet_last_error")))
    _torch_ext = rxmet_torch
    return rxmet_torch


def register(name: str, restype, argtypes) -> None:
    """Add a signature (used by modules that extend the ABI)."""
    _SIGNATURES[name] = (restype, argtypes)
    if _lib is not None:
        fn = getattr(_lib, name)
        fn.restype = restype
        fn.argtypes = argtypes


def call(name: str, *args) -> int:
    """Call ``name`` and raise RxmetError with the library's message on failure."""
    lib = load()
    rc = getattr(lib, name)(*args)
    if isinstance(rc, int) and rc != 0:
        msg = lib.rxmet_last_error().decode(errors="replace")
        raise RxmetError(f"{name} failed ({rc}): {msg}")
    return rc


def ptr(t) -> Optional[int]:
    """Device pointer of a tensor, or None for a missing optional argument."""
    return None if t is None else t.data_ptr()


def stream_of(device) -> int:
    """Handle of PyTorch's current HIP stream on ``device``."""
    import torch

    return torch.cuda.current_stream(device).cuda_stream


def block_copy(jobs, device) -> None:
    """Widen or narrow tensors in one launch (rxmet_block_copy): ``jobs`` holds (src, dst, outer,
    (rows_src, rows_dst), groups, (cols_src, cols_dst)) with contiguous fp32 tensors of exactly
    those sizes on ``device``."""
    import torch

    arr = (BlockJob * len(jobs))()
    for k, (src, dst, outer, rows, groups, cols) in enumerate(jobs):
        for t, r, c in ((src, rows[0], cols[0]), (dst, rows[1], cols[1])):
            if (t.dtype != torch.float32 or t.device != device or not t.is_contiguous()
                    or t.numel() != outer * r * groups * c):
                raise RuntimeError(f"block copy: a tensor of shape {tuple(t.shape)} ({t.dtype}, "
                                   f"{t.device}) is not [{outer}, {r}, {groups}, {c}] fp32")
        arr[k] = BlockJob(src.data_ptr(), dst.data_ptr(), outer, *rows, groups, *cols, 0)
    for k in range(0, len(jobs), BLOCK_JOBS):
        part = (BlockJob * min(BLOCK_JOBS, len(jobs) - k)).from_buffer(
            arr, k * ctypes.sizeof(BlockJob))
        call("rxmet_block_copy", len(part), part, stream_of(device))


def prof_enable(on: bool = True) -> None:
    """Turn the library's per-launch event timing on or off (include/rxmet_prof.h)."""
    load().rxmet_prof_enable(1 if on else 0)


def prof_filter(names=None) -> None:
    """Time only the named launches (an iterable of names; None: all)."""
    load().rxmet_prof_filter(None if names is None else ",".join(names).encode())


def prof_reset() -> None:
    load().rxmet_prof_reset()


def prof_query(name: str) -> tuple:
    """(total milliseconds, launches) recorded for an instrumented kernel name."""
    ms = ctypes.c_double(0.0)
    n = ctypes.c_int64(0)
    load().rxmet_prof_query(name.encode(), ctypes.byref(ms), ctypes.byref(n))
    return ms.value, n.value


def prof_names() -> list:
    lib = load()
    need = lib.rxmet_prof_names(None, 0)
    buf = ctypes.create_string_buffer(int(need) + 1)
    lib.rxmet_prof_names(buf, need + 1)
    return [n for n in buf.value.decode().split(",") if n]
