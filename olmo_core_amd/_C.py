"""
ctypes binding of libmi8.so (the C ABI declared in include/mi8.h).

The library is loaded once; it is never built from here and there is no fallback path: if the shared
object is missing, every operator raises ``MI8LibraryMissing`` with the build command.
"""

from __future__ import annotations

import ctypes
import threading
from ctypes import c_char_p, c_float, c_int, c_int32, c_int64, c_uint32, c_void_p, POINTER
from pathlib import Path
from typing import Optional

from .exceptions import MI8KernelError

import os

# MI8_LIBRARY overrides the in-tree location (e.g. to try a differently built library)
LIB_PATH = Path(os.environ.get("MI8_LIBRARY") or (Path(__file__).resolve().parent / "lib" / "libmi8.so"))

MI8_E4M3, MI8_E5M2 = 0, 1
MI8_BF16, MI8_F32, MI8_F16, MI8_RAW8, MI8_F32_OF_BF16 = 0, 1, 2, 3, 4
FLAG_POW2_SCALE = 1
FLAG_SW_CVT = 2
FLAG_AMAX_READY = 4
FLAG_PAD_T128 = 8
FLAG_READ_BY_FEW_ROWS = 16
AMAX_SLOTS = 2048

CAST_BATCH = 8


class CastItem(ctypes.Structure):
    """mi8_cast_item"""
    _fields_ = [("x", c_void_p), ("rows", c_int64), ("cols", c_int64), ("slots", c_void_p), ("scale_in", c_void_p),
                ("amax_ws", c_void_p), ("out", c_void_p), ("ld_out", c_int64), ("out_t", c_void_p), ("ld_t", c_int64),
                ("scale_out", c_void_p), ("n_slots", c_int32), ("hp_dtype", c_int32), ("pad_t128", c_int32)]


class TwoCastItem(ctypes.Structure):
    """mi8_two_cast_item"""
    _fields_ = [("x", c_void_p), ("rows", c_int64), ("cols", c_int64), ("out_rows", c_void_p), ("ld_rows", c_int64),
                ("row_scale", c_void_p), ("out_t", c_void_p), ("ld_t", c_int64), ("col_scale", c_void_p),
                ("workspace", c_void_p), ("group_rows", c_int64), ("hp_dtype", c_int32)]


GEMM_BATCH = 8


class GemmProduct(ctypes.Structure):
    """mi8_gemm_product"""
    _fields_ = [("a", c_void_p), ("lda", c_int64), ("b", c_void_p), ("ldb", c_int64), ("M", c_int64), ("N", c_int64),
                ("K", c_int64), ("sa", c_void_p), ("sb", c_void_p), ("out", c_void_p), ("ldc", c_int64),
                ("sa_is_vector", c_int32), ("sb_is_vector", c_int32), ("out_dtype", c_int32), ("add_to_previous", c_int32)]


# name -> (restype, argtypes); mirrors include/mi8.h one to one
_SIGNATURES = {
    "mi8_version": (c_int, []),
    "mi8_last_error": (c_char_p, []),
    "mi8_amax_partials": (c_int, [c_void_p, c_int, c_int64, c_void_p, POINTER(c_int32), c_void_p]),
    "mi8_amax_partials_batch": (c_int, [POINTER(c_void_p), POINTER(c_int64), c_int32, c_int, c_void_p, POINTER(c_int32), c_void_p]),
    "mi8_amax_slots_for": (c_int32, [c_int64]),
    "mi8_scale_from_partials": (c_int, [c_void_p, c_int32, c_int, c_uint32, c_void_p, c_void_p]),
    "mi8_multi_tensor_scales": (
        c_int,
        [c_void_p, c_void_p, c_int32, c_int, c_int, c_uint32, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_cast_tensorwise": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_void_p, c_int, c_uint32, c_void_p, c_int64,
         c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_cast_tensorwise_static": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_int, c_uint32, c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_cast_tensorwise_batch": (c_int, [POINTER(CastItem), c_int32, c_int, c_uint32, c_void_p]),
    "mi8_two_cast_workspace_words": (c_int64, [c_int64, c_int64]),
    "mi8_cast_rows_and_colwise_t_batch": (c_int, [POINTER(TwoCastItem), c_int32, c_int, c_uint32, c_void_p]),
    "mi8_cast_rowwise": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_int, c_uint32, c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_moe_sort_slots_max": (c_int64, []),
    "mi8_moe_sort_slots": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_moe_sort_workspace_words": (c_int64, [c_int64, c_int32]),
    "mi8_moe_sort_many_slots": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_moe_gather_cast_rows": (
        c_int,
        [c_void_p, c_int64, c_int64, c_void_p, c_int32, c_uint32, c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_swiglu_cast_rows": (
        c_int,
        [c_void_p, c_void_p, c_int64, c_int64, c_uint32, c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_colamax_workspace_slots": (c_int64, [c_int64, c_int64]),
    "mi8_cast_colwise_t": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_int, c_uint32, c_void_p, c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_gemm_fp8": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p,
         c_int, c_void_p, c_int, c_int64, c_int, c_void_p],
    ),
    "mi8_gemm_fp8_accumulate": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p,
         c_int, c_void_p, c_int, c_int64, c_void_p],
    ),
    "mi8_gemm_fp8_swiglu_matches_separate": (c_int, [c_int64, c_int64, c_int64]),
    "mi8_gemm_fp8_swiglu_pays": (c_int, [c_int64, c_int64, c_int64]),
    "mi8_gemm_fp8_swiglu": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_void_p, c_int, c_int64, c_int64, c_int64, c_int64, c_void_p, c_void_p,
         c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, POINTER(c_int32), c_void_p, c_void_p],
    ),
    "mi8_gemm_fp8_splitk": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p,
         c_int, c_void_p, c_int, c_int64, c_int, c_void_p, c_int64, c_void_p],
    ),
    "mi8_gemm_fp8_splitk_accumulate": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int, c_int64, c_int64, c_int64, c_int64, c_void_p, c_int, c_void_p,
         c_int, c_void_p, c_int, c_int64, c_int, c_void_p, c_int64, c_void_p],
    ),
    "mi8_gemm_fp8_batch_pays": (c_int, [POINTER(GemmProduct), c_int32]),
    "mi8_gemm_fp8_batch": (c_int, [POINTER(GemmProduct), c_int32, c_int, c_int, c_void_p]),
    "mi8_gemm_splitk_suggest": (c_int, [c_int64, c_int64, c_int64]),
    "mi8_gemm_splitk_workspace_bytes": (c_int64, [c_int64, c_int64, c_int]),
    "mi8_gemm_num_variants": (c_int, []),
    "mi8_gemm_variant_name": (c_char_p, [c_int]),
    "mi8_gemm_variant_for": (c_int, [c_int64, c_int64, c_int64, c_int, c_int]),
    "mi8_plan_function": (c_int, [c_char_p]),
    "mi8_run_plan": (c_int, [c_void_p, c_int64, c_void_p, c_int32, c_void_p]),
    "mi8_gemm_fp8_swiglu_slots": (c_int32, [c_int64, c_int64, c_int64]),
    "mi8_few_rows_swiglu_slots": (c_int32, [c_int64, c_int64, c_int64, c_int]),
    "mi8_few_rows_swiglu": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int64, c_void_p, c_void_p,
         c_uint32, c_void_p, c_void_p, POINTER(c_int32), c_void_p],
    ),
    "mi8_few_rows_cast_gemm": (
        c_int,
        [c_void_p, c_int64, c_void_p, c_int32, c_void_p, c_int64, c_int64, c_int64, c_int64, c_void_p, c_uint32, c_void_p,
         c_int64, c_void_p],
    ),
    "mi8_swiglu_fwd": (c_int, [c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p]),
    "mi8_swiglu_bwd": (
        c_int,
        [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_swiglu_bwd_cast": (
        c_int,
        [c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_void_p, c_int32, c_int, c_uint32, c_void_p, c_void_p,
         c_int64, c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_rowseg_code_count": (c_int64, [c_int64, c_int64]),
    "mi8_swiglu_amax_state_words": (c_int64, [c_int64, c_int64]),
    "mi8_rowseg_max_codes": (c_int, [c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_void_p]),
    "mi8_swiglu_bwd_amax_from_codes": (
        c_int,
        [c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_gemm_fp8_codes_supported": (c_int, [c_int64, c_int64, c_int64]),
    "mi8_gemm_fp8_codes": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int, c_int64, c_int64, c_int64, c_int64, c_void_p, c_void_p, c_void_p,
         c_int64, c_void_p, c_void_p],
    ),
    "mi8_moe_gather": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_void_p, c_int, c_int32, c_void_p, c_void_p],
    ),
    "mi8_moe_binned_gather": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_void_p, c_int, c_void_p, c_int32, c_int64, c_int32, c_void_p,
         c_void_p],
    ),
    "mi8_moe_scatter": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_void_p, c_int, c_int32, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_moe_binned_scatter": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_void_p, c_int, c_void_p, c_int32, c_int64, c_int32, c_void_p,
         c_void_p, c_void_p],
    ),
    "mi8_moe_scatter_wgrad": (
        c_int,
        [c_void_p, c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_void_p, c_void_p],
    ),
    "mi8_moe_binned_scatter_wgrad": (
        c_int,
        [c_void_p, c_void_p, c_int, c_int64, c_int64, c_void_p, c_void_p, c_int32, c_int64, c_int32, c_void_p, c_void_p],
    ),
    "mi8_grouped_padded_rows": (c_int64, [c_int64, c_int32]),
    "mi8_grouped_cast_colwise_t": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_int, c_uint32, c_void_p, c_void_p, c_int64, c_void_p,
         c_void_p],
    ),
    "mi8_grouped_swiglu_fwd": (
        c_int,
        [c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p],
    ),
    "mi8_grouped_swiglu_bwd": (
        c_int,
        [c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_int32, c_void_p, c_void_p, c_void_p, c_void_p,
         c_void_p, c_void_p, c_void_p],
    ),
    "mi8_grouped_cast_rows_and_colwise_t": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_int, c_uint32, c_void_p, c_void_p, c_int64, c_void_p,
         c_void_p, c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_moe_gather_cast_rows_and_colwise_t": (
        c_int,
        [c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_void_p, c_int, c_void_p, c_int32, c_int, c_uint32, c_void_p,
         c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_void_p],
    ),
    "mi8_grouped_gemm_fp8": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_int64, c_int64, c_int64,
         c_void_p, c_void_p, c_int64, c_void_p, c_int, c_int64, c_void_p],
    ),
    "mi8_grouped_gemm_fp8_accumulate": (
        c_int,
        [c_void_p, c_int, c_int64, c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_int64, c_int64, c_int64,
         c_void_p, c_void_p, c_int64, c_void_p, c_int, c_int64, c_void_p],
    ),
    "mi8_grouped_gemm_fp8_dual_supported": (c_int, [c_int64, c_int64, c_int64, c_int64]),
    "mi8_grouped_gemm_fp8_dual": (
        c_int,
        [c_void_p, c_void_p, c_int, c_int64, c_void_p, c_void_p, c_int, c_int64, c_int64, c_void_p, c_int32, c_int64, c_int64,
         c_int64, c_int64, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_void_p, c_int64, c_void_p],
    ),
    "mi8_grouped_wgrad_fp8": (
        c_int,
        [c_void_p, c_int, c_void_p, c_int, c_int64, c_void_p, c_int32, c_int64, c_int64, c_int64, c_void_p, c_void_p,
         c_void_p, c_int, c_void_p],
    ),
}

EXPORTED_SYMBOLS = tuple(_SIGNATURES)

# libmi8_diag.so (include/mi8_diag.h): measurement kernels and the plan of the persistent one, loaded by bench.py and tests only
DIAG_LIB_PATH = LIB_PATH.parent / "libmi8_diag.so"
_DIAG_SIGNATURES = {
    "mi8_diag_last_error": (c_char_p, []),
    "mi8_probe_mfma_loop": (c_int, [c_int, c_int, c_int, c_int, c_void_p, c_void_p]),
    "mi8_probe_mfma_feed": (c_int, [c_int, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p]),
    "mi8_probe_store_rate": (c_int, [c_int, c_int, c_int, c_int, c_void_p, c_int64, c_void_p, c_void_p]),
    "mi8_diag_gemm_tile_timeline": (c_int, [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int, c_int, c_void_p, c_void_p]),
    "mi8_diag_gemm_plan": (c_int, [c_int64, c_int64, c_int64, c_int, c_int, c_int, c_void_p]),
}
DIAG_EXPORTED_SYMBOLS = tuple(_DIAG_SIGNATURES)


class MI8LibraryMissing(RuntimeError):
    pass


_lib: Optional[ctypes.CDLL] = None

# per thread: what stands in for the library while a sequence of calls is recorded (float8/plan.py)
_recording = threading.local()


def lib() -> ctypes.CDLL:
    """The loaded library (loads on first use)."""
    global _lib
    recorder = getattr(_recording, "recorder", None)
    if recorder is not None:
        return recorder
    if _lib is None:
        if not LIB_PATH.exists():
            raise MI8LibraryMissing(
                f"{LIB_PATH} is not built. Build it with `python -m olmo_core_amd.build` (needs hipcc); "
                "there is no fallback implementation."
            )
        handle = ctypes.CDLL(str(LIB_PATH))
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = res
            fn.argtypes = args
        _lib = handle
    return _lib


_diag: Optional[ctypes.CDLL] = None


def diag() -> ctypes.CDLL:
    """The diagnostics library (loads on first use)."""
    global _diag
    if _diag is None:
        if not DIAG_LIB_PATH.exists():
            raise MI8LibraryMissing(f"{DIAG_LIB_PATH} is not built. Build it with `python -m olmo_core_amd.build`.")
        handle = ctypes.CDLL(str(DIAG_LIB_PATH))
        for name, (res, args) in _DIAG_SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = res
            fn.argtypes = args
        _diag = handle
    return _diag


def check_diag(status: int, what: str = "") -> None:
    if status != 0:
        msg = diag().mi8_diag_last_error()
        raise MI8KernelError(f"{what or 'libmi8_diag'}: error {status}: {msg.decode() if msg else ''}")


def is_built() -> bool:
    return LIB_PATH.exists()


def last_error() -> str:
    msg = lib().mi8_last_error()
    return msg.decode() if msg else ""


def check(status: int, what: str = "") -> None:
    """Raise on a non-zero status from the library."""
    if status != 0:
        kind = {-1: "bad argument", -2: "unsupported shape/alignment", -3: "launch failure"}.get(status, "error")
        raise MI8KernelError(f"{what or 'libmi8'}: {kind} ({status}): {last_error()}")
