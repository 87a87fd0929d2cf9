"""ctypes binding of ``libmoe_fused_linear.so`` (the gfx950 HIP library).

PyTorch supplies device memory and the current HIP stream; every computation on the
hot path happens in the library.  There is no fallback: if the shared object is absent
the first call raises, it never silently computes on another path.
"""
from __future__ import annotations

import ctypes
import os
from typing import Optional

import torch
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libmoe_fused_linear.so")
CSRC_DIR = os.path.normpath(os.path.join(_HERE, "..", "csrc"))

BF16, F32, F16 = 0, 1, 2
I32, I64 = 0, 1

_DTYPES = {torch.bfloat16: BF16, torch.float32: F32, torch.float16: F16}
_ITYPES = {torch.int32: I32, torch.int64: I64}

_vp, _i, _i64, _f, _sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_int64, ctypes.c_float, ctypes.c_size_t



class Nf4Weight(ctypes.Structure):
    """``mfl_nf4_weight``: a packed 4-bit matrix with its quantisation state, as device pointers."""

    _fields_ = [("packed", _vp), ("code16", _vp), ("absmax", _vp), ("absmax_tiled", _vp), ("absmax_u8", _vp),
                ("code256", _vp), ("absmax2", _vp), ("offset", _vp), ("blocksize", _i), ("blocksize2", _i)]


_nf4p = ctypes.POINTER(Nf4Weight)


class MoeBlock(ctypes.Structure):
    """``mfl_moe_block``: the sparse block after its router projection."""

    _fields_ = [("tokens", _vp), ("logits", _vp), ("w_gate", _vp), ("w_up", _vp), ("w_down", _vp), ("q_gate", _nf4p),
                ("q_up", _nf4p), ("q_down", _nf4p), ("T", _i64), ("E", _i), ("k", _i), ("H", _i), ("I", _i), ("renorm", _i),
                ("dtype", _i), ("logits_dtype", _i), ("training", _i)]


_blockp = ctypes.POINTER(MoeBlock)


class BlockCopy(ctypes.Structure):
    """``mfl_block_copy``: a strided copy of runs of bytes."""

    _fields_ = [("src", _vp), ("dst", _vp), ("blocks", _i64), ("bytes", _i64), ("src_stride", _i64), ("dst_stride", _i64)]


# name -> (restype, argtypes); mirrors include/moe_fused_linear.h
_SIGNATURES = {
    "mfl_abi_version": (_i, []),
    "mfl_strerror": (ctypes.c_char_p, [_i]),
    "mfl_gemm_fwd": (_i, [_vp, _vp, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _f, _i, _vp]),
    "mfl_gemm_dx": (_i, [_vp, _vp, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _f, _i, _vp]),
    "mfl_gemm_dw": (_i, [_vp, _vp, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _f, _i, _vp]),
    "mfl_gemm_dw_split_workspace": (_sz, [_i64, _i, _i, _i]),
    "mfl_gemm_dw_split": (_i, [_vp, _vp, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _f, _vp, _sz, _vp]),
    "mfl_gemm_fwd_nf4": (_i, [_vp, _vp, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_gemm_dx_nf4": (_i, [_vp, _vp, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _f, _i, _vp]),
    "mfl_gemm_dx_dual": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_gemm_dx_silu_bwd": (_i, [_vp, _vp, _vp, _vp, _vp, _i, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _vp]),
    "mfl_gemm_fwd_lora": (_i, [_vp, _vp, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_gemm_dx_lora": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_gemm_fwd_nf4_lora": (_i, [_vp, _vp, _vp, _vp, _i, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_gemm_dx_nf4_lora": (_i, [_vp, _vp, _vp, _vp, _i, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_gemm_fwd_gather": (_i, [_vp, _i64, _vp, _i, _vp, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_gemm_fwd_nf4_gather": (_i, [_vp, _i64, _vp, _i, _vp, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i,
                                     _vp]),
    "mfl_glu_fwd": (_i, [_vp, _i64, _vp, _i, _vp, _vp, _vp, _i, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _vp]),
    "mfl_glu_fwd_lora": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _i, _vp, _i, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _vp]),
    "mfl_glu_fwd_nf4": (_i, [_vp, _i64, _vp, _i, _vp, _vp, _vp, _i, _vp, _vp, _vp, _i, _vp, _i, _vp, _vp, _vp, _i64,
                             _i, _i, _i, _i, _vp]),
    "mfl_nf4_tiled_absmax_floats": (_i64, [_i, _i, _i, _i]),
    "mfl_nf4_tile_absmax": (_i, [_vp, _i, _i, _i, _i, _vp, _vp]),
    "mfl_gemm_fwd_nf4_tiled": (_i, [_vp, _i64, _vp, _i, _vp, _vp, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i,
                                    _i, _vp]),
    "mfl_glu_fwd_nf4_tiled": (_i, [_vp, _i64, _vp, _i, _vp, _vp, _vp, _vp, _i, _vp, _vp, _vp, _vp, _i, _vp, _i, _vp,
                                   _vp, _vp, _i64, _i, _i, _i, _i, _vp]),
    "mfl_gemm_fwd_nf4_packed": (_i, [_vp, _i64, _vp, _i, _nf4p, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_glu_fwd_nf4_packed": (_i, [_vp, _i64, _vp, _i, _nf4p, _nf4p, _vp, _i, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _vp]),
    "mfl_glu_fwd_nf4_lora": (_i, [_vp, _nf4p, _nf4p, _vp, _vp, _vp, _i, _vp, _i, _vp, _vp, _vp, _i64, _i, _i, _i, _i, _vp]),
    "mfl_gemm_dx_nf4_dual_lora": (_i, [_vp, _nf4p, _vp, _nf4p, _vp, _vp, _i, _vp, _i, _vp, _i64, _i, _i, _i, _i, _i, _vp]),
    "mfl_nf4_dequant": (_i, [_vp, _vp, _vp, _i, _vp, _i64, _i, _vp]),
    "mfl_dequant_blockwise_u8": (_i, [_vp, _vp, _vp, _i, _f, _vp, _i64, _vp]),
    "mfl_nf4_unnest_absmax": (_i, [_vp, _vp, _vp, _i, _vp, _vp, _i64, _vp]),
    "mfl_nf4_write_out_scales": (_i, [_nf4p, ctypes.POINTER(_i64), ctypes.POINTER(_vp), _i, _vp]),
    "mfl_nf4_quant": (_i, [_vp, _i, _i64, _i, _vp, _vp, _vp, _vp]),
    "mfl_router_fwd": (_i, [_vp, _vp, _vp, _i64, _i, _i, _i, _vp]),
    "mfl_router_dw_workspace": (_sz, [_i64, _i, _i]),
    "mfl_router_dw": (_i, [_vp, _vp, _vp, _i64, _i, _i, _vp, _sz, _vp]),
    "mfl_route_softmax_topk": (_i, [_vp, _i, _i64, _i, _i, _i, _vp, _vp, _i, _vp, _vp]),
    "mfl_route_softmax_topk_bwd": (_i, [_vp, _i, _i64, _i, _i, _i, _vp, _vp, _vp, _i, _vp, _vp]),
    "mfl_route_sort_small": (_i, [_vp, _i, _i64, _i, _i, _i, _vp, _vp, _i, _vp, _vp, _vp, _vp, _vp]),
    "mfl_route_sort_workspace": (_sz, [_i64, _i, _i]),
    "mfl_route_sort": (_i, [_vp, _i, _i64, _i, _i, _i, _vp, _vp, _i, _vp, _vp, _vp, _vp, _vp, _sz, _vp]),
    "mfl_expert_sort_workspace": (_sz, [_i64, _i]),
    "mfl_expert_sort": (_i, [_vp, _i, _i64, _i, _vp, _vp, _vp, _vp, _sz, _vp]),
    "mfl_expert_sort_static": (_i, [_vp, _i, _i64, _i, _vp, _vp, _vp, _vp]),
    "mfl_gather_rows": (_i, [_vp, _vp, _i, _vp, _vp, _i64, _i, _i, _vp]),
    "mfl_scatter_rows": (_i, [_vp, _vp, _i, _vp, _vp, _i64, _i, _i, _vp]),
    "mfl_combine_rows": (_i, [_vp, _vp, _vp, _vp, _i64, _i, _i, _i, _vp]),
    "mfl_copy_blocks": (_i, [ctypes.POINTER(BlockCopy), _i, _vp]),
    "mfl_rows_dot": (_i, [_vp, _vp, _vp, _vp, _i64, _i, _i, _i, _vp]),
    "mfl_silu_mul_fwd": (_i, [_vp, _vp, _vp, _i64, _i, _vp]),
    "mfl_silu_mul_bwd": (_i, [_vp, _vp, _vp, _vp, _vp, _vp, _i64, _i, _vp]),
    "mfl_moe_block_workspace": (_sz, [_blockp]),
    "mfl_moe_block_fwd": (_i, [_blockp, _vp, _vp, _sz, _vp]),
    "mfl_moe_block_bwd_workspace": (_sz, [_blockp]),
    "mfl_moe_block_bwd": (_i, [_blockp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _vp, _sz, _vp]),
}

# the entry points declared in include/moe_fused_linear.h: the library exports these and nothing else
ABI_SYMBOLS = tuple(_SIGNATURES)

_lib: Optional[ctypes.CDLL] = None


class MflError(RuntimeError):
    """A library entry point returned a non-zero status."""


def lib() -> ctypes.CDLL:
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise MflError(
                f"{LIB_PATH} is missing: build it with `make -C {CSRC_DIR}` (hipcc, gfx950). "
                "There is no fallback path."
            )
        handle = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype = res
            fn.argtypes = args
        if handle.mfl_abi_version() != 1:
            raise MflError("libmoe_fused_linear.so has an unexpected ABI version")
        _lib = handle
    return _lib


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = lib().mfl_strerror(rc).decode()
        raise MflError(f"{what} failed with status {rc}: {msg}")


def dtype_code(dt: torch.dtype) -> int:
    try:
        return _DTYPES[dt]
    except KeyError:
        raise TypeError(f"unsupported element type {dt}; expected bfloat16, float32 or float16") from None


def itype_code(dt: torch.dtype) -> int:
    try:
        return _ITYPES[dt]
    except KeyError:
        raise TypeError(f"unsupported index type {dt}; expected int32 or int64") from None


def ptr(t: Optional[torch.Tensor]) -> Optional[int]:
    return None if t is None else t.data_ptr()


# the current stream's handle without building a Stream object for it (4 us of every call)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_device = getattr(torch._C, "_cuda_getDevice", None)


def stream() -> int:
    if _raw_stream is None or _device is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_device())


# (bound once: the questions are asked in every call, and in a backward pass on another core than the forward's)
_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack
_transforms, _tracing_state = torch._C._functorch.peek_interpreter_stack, torch._C._get_tracing_state
_batched = torch._C._functorch.is_legacy_batchedtensor


def plain_gradient(grad: torch.Tensor) -> bool:
    """Whether a backward pass may hand this gradient's address to a kernel: no graph of the gradients is asked for, no
    transform or mode is watching, and it is not several gradients at once (batched tensors have no address)."""
    return not torch.is_grad_enabled() and _dispatch_modes() == 0 and _transforms() is None and not _batched(grad)


def plain_call() -> bool:
    """Whether a call that passes autograd by, or stands in for a stock operator, may do so: no forward-mode level, no
    functorch transform, no dispatch mode (counters, fake tensors, selective checkpointing) and no function mode (but for
    default devices, which watch nothing) that would have to see the operators, and nobody tracing or compiling (asked first: a compiler cannot look into the others)."""
    return (not torch.compiler.is_compiling() and forward_ad._current_level < 0 and _dispatch_modes() == 0
            and _transforms() is None and _tracing_state() is None
            and (_function_modes() == 0 or all(isinstance(torch._C._get_function_stack_at(i), DeviceContext)
                                               for i in range(_function_modes()))))


def dense(t: torch.Tensor) -> torch.Tensor:
    """``t.contiguous()``, asked first: the call gives the interpreter's lock away, and in a backward pass another thread
    wants it (up to 5 us each until it is back)."""
    return t if t.is_contiguous() else t.contiguous()


def as_index_tensor(m_sizes: torch.Tensor) -> torch.Tensor:
    """int32/int64 pass straight through; the narrower integer types the reference also
    accepts are widened on the device (no host sync)."""
    if m_sizes.dtype in _ITYPES:
        return m_sizes
    return m_sizes.to(torch.int32)
