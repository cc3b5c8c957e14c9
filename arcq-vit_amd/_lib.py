"""ctypes loader for ``libarcq_hip.so`` (the C ABI declared in ``include/arcq_hip.h``).

There is deliberately no fallback: if the shared library has not been built,
every op raises, so a GPU run can never silently go through something else.
"""
from __future__ import annotations

import ctypes
import os
import sys
import threading
import warnings

_PKG_DIR = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_PKG_DIR, "libarcq_hip.so")

ARCQ_F32 = 0
ARCQ_F16 = 1
ARCQ_STATIC_SCRATCH_BYTES = 40 * 1024 * 1024

_c_i64 = ctypes.c_int64
_c_int = ctypes.c_int
_c_ptr = ctypes.c_void_p
_c_f32 = ctypes.c_float

class LinearExArgs(ctypes.Structure):
    """``arcq_linear_ex_args`` of include/arcq_hip.h."""
    _fields_ = [("struct_size", ctypes.c_uint32),
                ("x_dtype", ctypes.c_int32), ("y_dtype", ctypes.c_int32), ("producer", ctypes.c_int32),
                ("activation", ctypes.c_int32), ("bits", ctypes.c_int32), ("group_size", ctypes.c_int32),
                ("ln_eps", ctypes.c_float),
                ("M", ctypes.c_int64), ("N", ctypes.c_int64), ("K", ctypes.c_int64),
                ("x", ctypes.c_void_p), ("ln_weight", ctypes.c_void_p), ("ln_bias", ctypes.c_void_p),
                ("a_thresholds", ctypes.c_void_p), ("a_codebook", ctypes.c_void_p), ("packed_w", ctypes.c_void_p),
                ("w_codebook", ctypes.c_void_p), ("w_center", ctypes.c_void_p), ("w_scale", ctypes.c_void_p),
                ("w_code_sum", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("residual", ctypes.c_void_p),
                ("x_hat_ws", ctypes.c_void_p), ("w_hat_ws", ctypes.c_void_p), ("y", ctypes.c_void_p),
                ("next_a_thresholds", ctypes.c_void_p), ("next_a_codebook", ctypes.c_void_p)]


class PrepareWeights(ctypes.Structure):
    """``arcq_prepare_weights`` of include/arcq_hip.h."""
    _fields_ = [(n, ctypes.c_void_p) for n in ("packed", "codebook", "center", "scale", "code_sum", "w_hat")] + [
        ("N", ctypes.c_int64), ("K", ctypes.c_int64), ("row_major", ctypes.c_int32), ("w_mult", ctypes.c_float)]


class PrepareArgs(ctypes.Structure):
    """``arcq_prepare_args``."""
    _fields_ = [("x_dtype", ctypes.c_int32), ("bits", ctypes.c_int32), ("ln_eps", ctypes.c_float), ("fp8", ctypes.c_int32),
                ("rows", ctypes.c_int64), ("K", ctypes.c_int64)] + [
        (n, ctypes.c_void_p) for n in ("x", "ln_weight", "ln_bias", "thresholds", "codebook", "x_hat")] + [
        ("weights", PrepareWeights * 2)]


class LinearPreparedArgs(ctypes.Structure):
    """``arcq_linear_prepared_args``."""
    _fields_ = [(n, ctypes.c_int32) for n in ("y_dtype", "activation", "next_bits", "w_row_major")] + [
        (n, ctypes.c_int64) for n in ("M", "N", "K")] + [
        (n, ctypes.c_void_p) for n in ("x_hat", "w_hat", "bias", "residual", "next_thresholds", "next_codebook", "y")] + [
        ("fp8", ctypes.c_int32), ("w_mult", ctypes.c_float)]


class LinearIndexArgs(ctypes.Structure):
    """``arcq_linear_index_args``."""
    _fields_ = [(n, ctypes.c_void_p) for n in ("x_codes", "x_center", "x_scale", "x_code_sum", "w_codes", "w_center", "w_scale",
                                               "w_code_sum", "product_table", "a_codebook", "w_codebook", "bias", "y")] + [
        (n, ctypes.c_int64) for n in ("rows", "out_features", "in_features")] + [
        (n, ctypes.c_int32) for n in ("bits", "group_size", "levels", "reserved")]


class MlpLayer(ctypes.Structure):
    """``arcq_mlp_layer``."""
    _fields_ = [(n, ctypes.c_void_p) for n in ("a_thresholds", "a_codebook", "packed_w", "w_codebook", "w_center", "w_scale",
                                               "w_code_sum", "bias", "w_hat_ws")]


class MlpArgs(ctypes.Structure):
    """``arcq_mlp_args``."""
    _fields_ = [("bits", ctypes.c_int32), ("eps", ctypes.c_float), ("ln_eps", ctypes.c_float)] + [
        (n, ctypes.c_int64) for n in ("M", "K", "H")] + [(n, ctypes.c_void_p) for n in ("x", "ln_weight", "ln_bias")] + [
        ("fc1", MlpLayer), ("fc2", MlpLayer), ("y", ctypes.c_void_p), ("attn", ctypes.c_void_p), ("proj", MlpLayer)]


ARCQ_PRODUCER_NONE, ARCQ_PRODUCER_LAYERNORM, ARCQ_PRODUCER_XHAT = 0, 1, 2
ARCQ_ACT_NONE, ARCQ_ACT_GELU = 0, 1

# name -> argtypes, in the order of include/arcq_hip.h
_SIGNATURES = {
    "arcq_pack_codes": [_c_ptr, _c_ptr, _c_i64, _c_i64, _c_int, _c_ptr],
    "arcq_unpack_codes": [_c_ptr, _c_ptr, _c_i64, _c_i64, _c_int, _c_ptr],
    "arcq_unpack_codes_u8": [_c_ptr, _c_ptr, _c_i64, _c_i64, _c_int, _c_ptr],
    "arcq_act_quant": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_int,
                       _c_i64, _c_i64, _c_int, _c_int, _c_f32, _c_ptr],
    "arcq_weight_dequant": [_c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_int, _c_i64, _c_i64, _c_int, _c_int,
                            _c_ptr],
    "arcq_linear_fused": [_c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_int,
                          _c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_ptr],
    "arcq_linear_otf": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr,
                        _c_ptr, _c_int, _c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_ptr],
    "arcq_linear_fused_ws": [_c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_int,
                             _c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_ptr],
    "arcq_linear_otf_ws": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr,
                           _c_ptr, _c_ptr, _c_int, _c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_ptr],
    "arcq_linear_otf_static": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr,
                               _c_ptr, _c_int, _c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_ptr],
    "arcq_linear_otf_ex": [ctypes.POINTER(LinearExArgs), _c_ptr],
    "arcq_xhat_layout": [_c_i64],
    "arcq_prepared_row_major": [_c_i64, _c_i64, _c_i64],
    "arcq_prepared_quant_row_major": [_c_i64, _c_i64, _c_i64, _c_int],
    "arcq_prepare_patches": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_int, _c_f32,
                             ctypes.POINTER(PrepareWeights), _c_ptr],
    "arcq_prepare": [ctypes.POINTER(PrepareArgs), _c_ptr],
    "arcq_linear_prepared": [ctypes.POINTER(LinearPreparedArgs), _c_ptr],
    "arcq_mlp_otf": [ctypes.POINTER(MlpArgs), _c_ptr],
    "arcq_mlp_otf_supported": [_c_i64, _c_i64, _c_i64],
    "arcq_mlp_otf_pays": [_c_i64, _c_i64, _c_i64],
    "arcq_act_quant_blocked_ln": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_f32, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_int,
                                  _c_f32, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_ptr],
    "arcq_act_quant_blocked": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_int, _c_f32, _c_ptr],
    "arcq_act_quant_fp8": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_int, _c_f32, _c_ptr],
    "arcq_weight_dequant_fp8": [_c_ptr] * 6 + [_c_i64, _c_i64, _c_int, _c_int, _c_f32, _c_ptr],
    "arcq_act_quant_fp8_blocked": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_int, _c_f32,
                                   _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_f32, _c_ptr],
    "arcq_linear_fp8_blocked": [_c_ptr, _c_ptr, _c_ptr, _c_f32, _c_ptr, _c_int, _c_i64, _c_i64, _c_i64, _c_ptr],
    "arcq_linear_otf_fp8": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_f32,
                            _c_ptr, _c_ptr, _c_ptr, _c_int, _c_i64, _c_i64, _c_i64, _c_int, _c_ptr],
    "arcq_act_quant_blocked_with_weights": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_int, _c_f32,
                                            _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_ptr],
    "arcq_linear_fused_blocked": [_c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_int, _c_ptr, _c_int,
                                  _c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_ptr],
    "arcq_act_quant_patches": [_c_ptr, _c_int, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_int, _c_f32,
                               _c_int, _c_ptr],
    "arcq_patch_embed_fwd": [_c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_ptr, _c_i64, _c_i64, _c_i64, _c_i64, _c_i64, _c_ptr],
    "arcq_attention_quant_fwd": [_c_ptr, _c_ptr, _c_ptr, _c_int, _c_ptr, _c_i64, _c_i64, _c_i64, _c_i64, _c_f32, _c_ptr],
    "arcq_attention_quant_fp8_fwd": [_c_ptr, _c_ptr, _c_ptr, _c_int, _c_ptr, _c_i64, _c_i64, _c_i64, _c_i64, _c_f32, _c_ptr],
    "arcq_attention_fwd": [_c_ptr, _c_ptr, _c_i64, _c_i64, _c_i64, _c_i64, _c_f32, _c_ptr],
    "arcq_linear_index": [ctypes.POINTER(LinearIndexArgs), _c_ptr],
    "arcq_linear_forward_packed": [_c_ptr] * 11 + [_c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_int, _c_ptr],
    "arcq_linear_forward_u8": [_c_ptr] * 11 + [_c_i64, _c_i64, _c_i64, _c_int, _c_int, _c_ptr],
}
EXPORTED_SYMBOLS = ("arcq_version", "arcq_last_error", "arcq_reload_tuning", "arcq_linear_fused_kernel",
                    "arcq_linear_fused_ws_kernel", "arcq_linear_otf_ws_kernel", "arcq_rows_wait_timeouts",
                    "arcq_rows_counter_slot") + tuple(_SIGNATURES)

_lib = None
_lock = threading.Lock()


class ARCQLibraryMissing(ImportError):
    pass


def load() -> ctypes.CDLL:
    """Load the library once; raise if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is None:
            if not os.path.exists(LIB_PATH):
                raise ARCQLibraryMissing(
                    f"ARCQ HIP library is not built ({LIB_PATH} missing). "
                    "Run `python -m arcq_vit_amd.build` (needs hipcc) first.")
            lib = ctypes.CDLL(LIB_PATH)
            lib.arcq_version.restype = _c_int
            lib.arcq_version.argtypes = []
            lib.arcq_last_error.restype = ctypes.c_char_p
            lib.arcq_last_error.argtypes = []
            lib.arcq_reload_tuning.restype = None
            lib.arcq_reload_tuning.argtypes = []
            lib.arcq_linear_fused_kernel.restype = ctypes.c_char_p
            lib.arcq_linear_fused_kernel.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64]
            lib.arcq_linear_fused_ws_kernel.restype = ctypes.c_char_p
            lib.arcq_linear_fused_ws_kernel.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
            lib.arcq_linear_otf_ws_kernel.restype = ctypes.c_char_p
            lib.arcq_linear_otf_ws_kernel.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
            lib.arcq_rows_wait_timeouts.restype = ctypes.c_longlong
            lib.arcq_rows_wait_timeouts.argtypes = []
            lib.arcq_rows_counter_slot.restype = _c_int
            lib.arcq_rows_counter_slot.argtypes = [ctypes.POINTER(ctypes.c_void_p), _c_int, _c_ptr]
            for name, argtypes in _SIGNATURES.items():
                fn = getattr(lib, name)
                fn.restype = _c_int
                fn.argtypes = argtypes
            _lib = lib
    return _lib


_host = None


class _NoHost:
    """In the place of the host extension where that does not load: every call is left to the Python code behind it."""

    def _leave(*args):
        return None

    layer_forward = block_forward = attention = patch_embed = quantize = packed_forward = patch_conv_forward = _leave


def host():
    """The CPython extension with the host side of the hot calls (``csrc_host/arcq_host.cpp``).  Its functions return None for
    calls they leave to the Python code.  It is built against one torch; where it does not load, the same kernels are called
    through ctypes (slower in host time and, for whole blocks, in launches), which is said once.  Without the library itself
    this raises, as ``load`` does."""
    global _host
    if _host is None:
        load()
        try:
            from . import _arcq_host as mod
        except ImportError as e:
            warnings.warn(f"ARCQ host extension is not built or does not load ({e}); the kernels are called through ctypes, which "
                          "is slower. Run `python -m arcq_vit_amd.build` to build it.", RuntimeWarning, stacklevel=3)
            _host = _NoHost
            return _host
        import torch
        from . import ops, vit
        from .packed_on_the_fly import ARCQPackedLinearOnTheFly
        mod.register_types(ARCQPackedLinearOnTheFly, vit.Attention, vit.Mlp, torch.nn.GELU, torch.nn.LayerNorm,
                           sys.modules["torch.nn.modules.module"], ops.fp8_weight_multiplier)
        _host = mod
    return _host


def host_for_block():
    """``host()`` for a module that need not hold a packed layer: it runs without the library too."""
    if _host is None and not os.path.exists(LIB_PATH):
        return _NoHost
    return host()


def check(rc: int) -> None:
    """Raise ``RuntimeError`` for a non-zero return, as ``TORCH_CHECK`` does in the reference's
    host wrappers (e.g. EXT/arcq_activation_kernel.cu:194-202)."""
    if rc != 0:
        msg = load().arcq_last_error().decode("utf-8", "replace")
        raise RuntimeError(msg or f"libarcq_hip call failed with code {rc}")


def reload_tuning() -> None:
    """Make the library read its ``ARCQ_*`` tuning variables again (it reads them once per process)."""
    load().arcq_reload_tuning()
