"""Binding of libfmsa_hip.so (C ABI declared in include/fmsa.h): the calls of the operators' hot path through the extension
built from csrc/host_calls.cpp, everything else through ctypes.

Both are built in-tree by ``build_hip.py`` and loaded from ``../lib``.  Nothing here falls
back to another implementation: if the library is missing, or a call returns an error code, a
RuntimeError is raised.  torch is used only for device memory (tensors) and the current stream.
"""
from __future__ import annotations

import ctypes
import importlib.util
import os
from ctypes import POINTER, Structure, c_float, c_int, c_int32, c_int64, c_size_t, c_void_p
from typing import Optional, Sequence

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(os.path.dirname(_HERE), "lib", "libfmsa_hip.so")
CALLS_PATH = os.path.join(os.path.dirname(_HERE), "lib", "_fmsa_calls.so")

F16, BF16, F32 = 0, 1, 2
FWD_LINEAR, FWD_SWIGLU = 0, 1
BWD_LINEAR, BWD_SWIGLU = 0, 1

_DTYPE_ENUM = {torch.float16: F16, torch.bfloat16: BF16, torch.float32: F32}

EXPORTED_SYMBOLS = (
    "fmsa_strerror",
    "fmsa_abi_version",
    "fmsa_gptq_dequant",
    "fmsa_gptq_permute_rows",
    "fmsa_permute_cols",
    "fmsa_lora_down",
    "fmsa_lora_down_workspace",
    "fmsa_lora_down_ws",
    "fmsa_lora_down_split_workspace",
    "fmsa_lora_down_split",
    "fmsa_lora_down_batch_workspace",
    "fmsa_lora_down_batch",
    "fmsa_lora_grad_workspace",
    "fmsa_lora_grad",
    "fmsa_lora_grad_batch_workspace",
    "fmsa_lora_grad_batch",
    "fmsa_lora_grad_static",
    "fmsa_gptq_lora_fwd",
    "fmsa_gptq_lora_fwd_workspace",
    "fmsa_gptq_lora_fwd_ws",
    "fmsa_gptq_lora_fwd_is_few",
    "fmsa_gptq_lora_fwd_few",
    "fmsa_lora_few_is_few",
    "fmsa_lora_few_workspace",
    "fmsa_lora_few_fwd",
    "fmsa_gptq_lora_fwd_rope",
    "fmsa_gptq_lora_fwd_rope_pays",
    "fmsa_gptq_lora_fwd_tile",
    "fmsa_gptq_lora_bwd_dx_tile",
    "fmsa_gptq_lora_bwd_dx",
    "fmsa_gptq_lora_bwd_dx_workspace",
    "fmsa_gptq_lora_bwd_dx_ws",
    "fmsa_swiglu_fwd",
    "fmsa_swiglu_bwd",
    "fmsa_gptq_make_nsz",
    "fmsa_gptq_transpose",
    "fmsa_gptq_interleave",
    "fmsa_nf4_dequant",
    "fmsa_nf4_prepare",
    "fmsa_lora_pack",
    "fmsa_lora_pack_batch",
    "fmsa_rms_layernorm_fwd",
    "fmsa_rms_layernorm_bwd",
    "fmsa_rope_embedding",
    "fmsa_rope_embedding_pair",
    "fmsa_rope_embedding_strided",
    "fmsa_cross_entropy_fwd",
    "fmsa_cross_entropy_bwd",
    "fmsa_cross_entropy_rows_fwd",
    "fmsa_cross_entropy_rows_fwd_keep",
    "fmsa_cross_entropy_rows_bwd",
    "fmsa_causal_lm_loss_workspace",
    "fmsa_causal_lm_loss_fwd",
    "fmsa_causal_lm_loss_bwd",
    "fmsa_cross_entropy_fused",
)


class GptqWeight(Structure):
    _fields_ = [
        ("qweight", c_void_p),
        ("scales", c_void_p),
        ("qzeros", c_void_p),
        ("g_idx", c_void_p),
        ("K", c_int32),
        ("N", c_int32),
        ("group_size", c_int32),
        ("zero_offset", c_int32),
        ("format", c_int32),
        ("nibble_order", c_int32),
        ("code", c_void_p),
        ("block_scale", c_void_p),
    ]


WEIGHT_AFFINE, WEIGHT_CODEBOOK = 0, 1


class Rope(Structure):
    _fields_ = [
        ("cos", c_void_p),
        ("sin", c_void_p),
        ("ld", c_int64),
        ("rows", c_int32),
        ("head_dim", c_int32),
        ("dtype", c_int32),
        ("proj_mask", c_int32),
    ]


class Nf4Weight(Structure):
    _fields_ = [
        ("packed", c_void_p),
        ("absmax_q", c_void_p),
        ("absmax2", c_void_p),
        ("code2", c_void_p),
        ("code", c_void_p),
        ("offset", c_float),
        ("N", c_int32),
        ("K", c_int32),
        ("blocksize", c_int32),
        ("blocksize2", c_int32),
    ]


class LoraGradJob(Structure):
    """fmsa_lora_grad_job: one scale * L[M, r]^T @ R[M, C] of a batch."""

    _fields_ = [
        ("L", c_void_p),
        ("R", c_void_p),
        ("out", c_void_p),
        ("ldl", c_int64),
        ("ldr", c_int64),
        ("C", c_int32),
        ("r", c_int32),
        ("scale", c_float),
        ("transpose_out", c_int32),
        ("out_dtype", c_int32),
        ("reserved", c_int32),
        ("Wt", c_void_p),
        ("T", c_void_p),
        ("ldt", c_int64),
    ]


class LoraDownJob(Structure):
    """fmsa_lora_down_job: one product of a batch."""

    _fields_ = [
        ("X", c_void_p),
        ("Wd", c_void_p),
        ("out", c_void_p),
        ("ldx", c_int64),
        ("ldout", c_int64),
        ("C", c_int32),
        ("r", c_int32),
    ]


class LoraPackJob(Structure):
    """fmsa_lora_pack_job: one adapter of a batched pack."""

    _fields_ = [
        ("A", c_void_p),
        ("B", c_void_p),
        ("A16", c_void_p),
        ("At16", c_void_p),
        ("B16", c_void_p),
        ("Bt16", c_void_p),
        ("r", c_int32),
        ("K", c_int32),
        ("N", c_int32),
        ("param_dtype", c_int32),
    ]


class FwdProj(Structure):
    _fields_ = [
        ("w", GptqWeight),
        ("U", c_void_p),
        ("ldu", c_int64),
        ("B", c_void_p),
        ("bias", c_void_p),
        ("Y", c_void_p),
        ("ldy", c_int64),
        ("r", c_int32),
        ("s", c_float),
    ]


class FewProj(Structure):
    _fields_ = [
        ("w", GptqWeight),
        ("A", c_void_p),
        ("B", c_void_p),
        ("bias", c_void_p),
        ("Y", c_void_p),
        ("ldy", c_int64),
        ("r", c_int32),
        ("s", c_float),
        ("param_dtype", c_int32),
        ("reserved", c_int32),
    ]


class BwdProj(Structure):
    _fields_ = [
        ("w", GptqWeight),
        ("nsz", c_void_p),
        ("dY", c_void_p),
        ("lddy", c_int64),
        ("T", c_void_p),
        ("ldt", c_int64),
        ("At", c_void_p),
        ("mask_src", c_void_p),
        ("ldmask", c_int64),
        ("r", c_int32),
        ("s", c_float),
        ("qweight_t", c_void_p),
        ("scale_f32", c_void_p),
        ("negzp_f16", c_void_p),
    ]


_lib = None


ABI_VERSION = 11  # include/fmsa.h as this binding mirrors it (fmsa_abi_version of the library must agree)


def lib() -> ctypes.CDLL:
    """The loaded library; raises if it has not been built."""
    global _lib
    if _lib is not None:
        return _lib
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(
            f"{LIB_PATH} is missing: build it with `python fms-acceleration_amd/build_hip.py` "
            "(there is no fallback path for the fused quantised-LoRA kernels)"
        )
    L = ctypes.CDLL(LIB_PATH)
    L.fmsa_strerror.restype = ctypes.c_char_p
    L.fmsa_strerror.argtypes = [c_int]
    L.fmsa_abi_version.restype = c_int
    if L.fmsa_abi_version() != ABI_VERSION:
        # struct layouts and signatures below are those of ABI_VERSION: a library of another version would read them wrong
        raise RuntimeError(f"{LIB_PATH} has ABI version {L.fmsa_abi_version()}, this binding is written for {ABI_VERSION}: "
                           "rebuild it with `python fms-acceleration_amd/build_hip.py`")
    L.fmsa_gptq_dequant.argtypes = [POINTER(GptqWeight), c_int, c_void_p, c_void_p]
    L.fmsa_gptq_permute_rows.argtypes = [c_void_p, c_void_p, c_int, c_int, c_void_p, c_void_p]
    L.fmsa_permute_cols.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_int64, c_void_p]
    L.fmsa_lora_down.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_int64, c_void_p]
    L.fmsa_lora_down_workspace.restype = c_size_t
    L.fmsa_lora_down_workspace.argtypes = [c_int, c_int, c_int]
    L.fmsa_lora_down_ws.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_int64, c_void_p, c_size_t,
                                    c_void_p]
    L.fmsa_lora_down_split_workspace.restype = c_size_t
    L.fmsa_lora_down_split_workspace.argtypes = [c_int, c_int, c_int]
    L.fmsa_lora_down_split.argtypes = L.fmsa_lora_down_ws.argtypes
    L.fmsa_lora_down_batch_workspace.restype = c_size_t
    L.fmsa_lora_down_batch_workspace.argtypes = [POINTER(LoraDownJob), c_int, c_int]
    L.fmsa_lora_down_batch.argtypes = [POINTER(LoraDownJob), c_int, c_int, c_int, c_void_p, c_size_t, c_void_p]
    L.fmsa_lora_grad_workspace.restype = c_size_t
    L.fmsa_lora_grad_workspace.argtypes = [c_int, c_int, c_int]
    L.fmsa_lora_grad.argtypes = [c_void_p, c_int64, c_void_p, c_int64, c_int, c_int, c_int, c_float, c_int, c_int, c_int,
                                 c_void_p, c_void_p, c_size_t, c_void_p]
    L.fmsa_lora_grad_batch_workspace.restype = c_size_t
    L.fmsa_lora_grad_batch_workspace.argtypes = [POINTER(LoraGradJob), c_int, c_int]
    L.fmsa_lora_grad_batch.argtypes = [POINTER(LoraGradJob), c_int, c_int, c_int, c_void_p, c_size_t, c_void_p]
    L.fmsa_lora_grad_static.argtypes = [c_void_p, c_int64, c_void_p, c_int64, c_int, c_int, c_int, c_float, c_int, c_int, c_int,
                                        c_void_p, c_void_p]
    L.fmsa_gptq_lora_fwd.argtypes = [POINTER(FwdProj), c_int, c_void_p, c_int64, c_int, c_int, c_void_p, c_int64,
                                     c_int, c_void_p]
    L.fmsa_gptq_lora_fwd_workspace.restype = c_size_t
    L.fmsa_gptq_lora_fwd_workspace.argtypes = [POINTER(FwdProj), c_int, c_int, c_int]
    L.fmsa_gptq_lora_fwd_ws.argtypes = [POINTER(FwdProj), c_int, c_void_p, c_int64, c_int, c_int, c_void_p, c_int64, c_int, c_void_p,
                                        c_size_t, c_void_p]
    L.fmsa_gptq_lora_fwd_is_few.argtypes = [POINTER(FwdProj), c_int, c_int, c_int]
    L.fmsa_gptq_lora_fwd_rope_pays.argtypes = [POINTER(FwdProj), c_int, c_int]
    L.fmsa_gptq_lora_fwd_tile.argtypes = [POINTER(FwdProj), c_int, c_int, c_int]
    L.fmsa_gptq_lora_bwd_dx_tile.argtypes = [POINTER(BwdProj), c_int, c_int, c_int, c_int]
    L.fmsa_gptq_lora_fwd_few.argtypes = L.fmsa_gptq_lora_fwd.argtypes
    L.fmsa_lora_few_is_few.argtypes = [POINTER(FewProj), c_int, c_int, c_int]
    L.fmsa_lora_few_workspace.restype = c_size_t
    L.fmsa_lora_few_workspace.argtypes = [POINTER(FewProj), c_int, c_int]
    L.fmsa_lora_few_fwd.argtypes = [POINTER(FewProj), c_int, c_void_p, c_int64, c_int, c_int, c_void_p, c_int64, c_int, c_void_p,
                                    c_size_t, c_void_p]
    L.fmsa_gptq_lora_bwd_dx_workspace.restype = c_size_t
    L.fmsa_gptq_lora_bwd_dx_workspace.argtypes = [POINTER(BwdProj), c_int, c_int, c_int]
    L.fmsa_gptq_lora_bwd_dx_ws.argtypes = [POINTER(BwdProj), c_int, c_int, c_int, c_void_p, c_int64, c_void_p, c_void_p, c_void_p,
                                           c_int64, c_int, c_void_p, c_size_t, c_void_p]
    L.fmsa_gptq_lora_fwd_rope.argtypes = [POINTER(FwdProj), c_int, c_void_p, c_int64, c_int, POINTER(Rope), c_int, c_void_p]
    L.fmsa_gptq_lora_bwd_dx.argtypes = [POINTER(BwdProj), c_int, c_int, c_int, c_void_p, c_int64, c_void_p, c_void_p,
                                        c_void_p, c_int64, c_int, c_void_p]
    L.fmsa_swiglu_fwd.argtypes = [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int64, c_int, c_void_p]
    L.fmsa_swiglu_bwd.argtypes = [c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int64, c_int, c_void_p]
    L.fmsa_gptq_make_nsz.argtypes = [POINTER(GptqWeight), c_void_p, c_void_p]
    L.fmsa_gptq_transpose.argtypes = [c_void_p, c_int, c_int, c_void_p, c_void_p]
    L.fmsa_gptq_interleave.argtypes = [c_void_p, c_int, c_int, c_void_p, c_void_p]
    L.fmsa_nf4_dequant.argtypes = [POINTER(Nf4Weight), c_int, c_void_p, c_void_p]
    L.fmsa_nf4_prepare.argtypes = [POINTER(Nf4Weight), c_void_p, c_void_p, c_void_p]
    L.fmsa_lora_pack.argtypes = [c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p,
                                 c_void_p]
    L.fmsa_lora_pack_batch.argtypes = [POINTER(LoraPackJob), c_int, c_int, c_void_p]
    L.fmsa_rms_layernorm_fwd.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_int, c_float, c_int, c_int, c_int, c_void_p,
                                         c_int64, c_void_p, c_void_p]
    L.fmsa_rms_layernorm_bwd.argtypes = [c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                                         c_int, c_void_p]
    L.fmsa_rope_embedding.argtypes = [c_void_p, c_int64, c_void_p, c_void_p, c_int64, c_int, c_int, c_int, c_int, c_int, c_int,
                                      c_int, c_void_p]
    L.fmsa_rope_embedding_pair.argtypes = [c_void_p, c_int64, c_int, c_void_p, c_int64, c_int, c_void_p, c_void_p, c_int64, c_int, c_int,
                                           c_int, c_int, c_int, c_int, c_void_p]
    L.fmsa_rope_embedding_strided.argtypes = [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_void_p, c_void_p, c_int64, c_int, c_int,
                                              c_int, c_int, c_int, c_int, c_int, c_int, c_void_p]
    L.fmsa_cross_entropy_fwd.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p]
    L.fmsa_cross_entropy_bwd.argtypes = [c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p]
    L.fmsa_cross_entropy_rows_fwd.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p]
    L.fmsa_cross_entropy_rows_fwd_keep.argtypes = [c_void_p, c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_int, c_int, c_void_p,
                                                   c_void_p, c_void_p]
    L.fmsa_cross_entropy_rows_bwd.argtypes = [c_void_p, c_void_p, c_int64, c_void_p, c_int64, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                                              c_int, c_void_p]
    L.fmsa_causal_lm_loss_workspace.restype = c_size_t
    L.fmsa_causal_lm_loss_workspace.argtypes = [c_int, c_int, c_int]
    L.fmsa_causal_lm_loss_fwd.argtypes = [c_void_p, c_void_p, c_int64, c_void_p, c_int64, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p,
                                          c_void_p, c_void_p, c_void_p, c_void_p, c_size_t, c_void_p]
    L.fmsa_causal_lm_loss_bwd.argtypes = [c_void_p, c_void_p, c_int64, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                                          c_int, c_void_p]
    L.fmsa_cross_entropy_fused.argtypes = [c_void_p, c_int64, c_void_p, c_int, c_int, c_int, c_int64, c_void_p, c_float, c_void_p, c_void_p]
    for name in EXPORTED_SYMBOLS:
        getattr(L, name)  # AttributeError here means the library is stale: rebuild it
    _lib = L
    return L


class FmsaError(RuntimeError):
    def __init__(self, fn: str, code: int):
        msg = lib().fmsa_strerror(code).decode()
        super().__init__(f"{fn} failed with code {code}: {msg}")
        self.code = code


_native = None


def native():
    """The extension of csrc/host_calls.cpp; raises if it has not been built."""
    global _native
    if _native is None:
        lib()
        if not os.path.exists(CALLS_PATH):
            raise RuntimeError(f"{CALLS_PATH} is missing: build it with `python fms-acceleration_amd/build_hip.py`")
        spec = importlib.util.spec_from_file_location("_fmsa_calls", CALLS_PATH)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        if module.install(FmsaError) != ABI_VERSION:
            raise RuntimeError(f"{CALLS_PATH} was built for another ABI version than {ABI_VERSION}, that of {LIB_PATH}: rebuild both")
        module.install_types(torch.nn.Identity, torch.nn.ModuleDict, torch.nn.Parameter)
        _native = module
    return _native


def _check(fn: str, code: int):
    if code != 0:
        raise FmsaError(fn, code)


# Pointers and streams go to ctypes as plain integers (it makes its own c_void_p from the argument types) and the stream is
# asked for by its raw handle, without a Stream object per launch.
def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _raw_stream(index: int) -> int:
    return torch._C._cuda_getCurrentRawStream(index)  # pylint: disable=protected-access


def _stream(t: torch.Tensor):
    if not t.is_cuda:
        raise RuntimeError("libfmsa_hip kernels need tensors on the GPU (there is no CPU implementation)")
    return _raw_stream(t.get_device())


def act_enum(dtype: torch.dtype) -> int:
    if dtype not in (torch.float16, torch.bfloat16):
        raise TypeError(f"activations must be float16 or bfloat16, got {dtype}")
    return _DTYPE_ENUM[dtype]


def make_weight(qweight, scales, qzeros, g_idx, group_size: int, zero_offset: int = 0, nibble_order: int = 0) -> GptqWeight:
    """GptqWeight from QuantLinear buffers.  g_idx=None declares the identity assignment.  nibble_order=1 declares
    that qweight is gptq_interleave's output (forward entry point, fp16 activations, group_size % 64 == 0 only)."""
    K = qweight.shape[0] * 8
    N = qweight.shape[1]
    assert qweight.dtype == torch.int32 and qzeros.dtype == torch.int32 and scales.dtype == torch.float16
    assert qweight.is_contiguous() and qzeros.is_contiguous() and scales.is_contiguous()
    return GptqWeight(
        qweight.data_ptr(), scales.data_ptr(), qzeros.data_ptr(),
        None if g_idx is None else g_idx.data_ptr(), K, N, int(group_size), int(zero_offset), WEIGHT_AFFINE, int(nibble_order), None, None,
    )


def make_codebook_weight(qweight, code, block_scale, group_size: int) -> GptqWeight:
    """GptqWeight of a 4-bit code-book weight in the word layout (what nf4_prepare returns):
    W[k, n] = code[q[k, n]] * block_scale[k // group_size, n]."""
    K, N = qweight.shape[0] * 8, qweight.shape[1]
    assert qweight.dtype == torch.int32 and code.dtype == torch.float32 and block_scale.dtype == torch.float32
    assert qweight.is_contiguous() and code.is_contiguous() and block_scale.is_contiguous()
    assert code.numel() == 16 and block_scale.shape == (K // group_size, N)
    return GptqWeight(qweight.data_ptr(), None, None, None, K, N, int(group_size), 0, WEIGHT_CODEBOOK, 0,
                      code.data_ptr(), block_scale.data_ptr())


def weight_dequant(w: GptqWeight, device, out_dtype=torch.float16):
    """Dense [K, N] of any GptqWeight (affine or code-book), one rounding to out_dtype."""
    out = torch.empty((w.K, w.N), dtype=out_dtype, device=device)
    _check("fmsa_gptq_dequant", lib().fmsa_gptq_dequant(ctypes.byref(w), _DTYPE_ENUM[out_dtype], _ptr(out), _stream(out)))
    return out


# ---- thin tensor-level wrappers ------------------------------------------------------------------
def gptq_dequant(qweight, scales, qzeros, g_idx, group_size, zero_offset=0, out_dtype=torch.float16):
    """W [K, N] = scales[g] * (q - z - zero_offset), one RNE rounding to out_dtype."""
    w = make_weight(qweight, scales, qzeros, g_idx, group_size, zero_offset)
    out = torch.empty((w.K, w.N), dtype=out_dtype, device=qweight.device)
    _check("fmsa_gptq_dequant", lib().fmsa_gptq_dequant(ctypes.byref(w), _DTYPE_ENUM[out_dtype], _ptr(out), _stream(out)))
    return out


def gptq_make_nsz(w: GptqWeight, device) -> torch.Tensor:
    """fp32 [G, N] table -scale * (zero + zero_offset) read by the input-gradient kernel."""
    G = (w.K + w.group_size - 1) // w.group_size
    out = torch.empty((G, w.N), dtype=torch.float32, device=device)
    _check("fmsa_gptq_make_nsz", lib().fmsa_gptq_make_nsz(ctypes.byref(w), _ptr(out), _stream(out)))
    return out


def gptq_permute_rows(qweight, perm):
    K, N = qweight.shape[0] * 8, qweight.shape[1]
    out = torch.empty_like(qweight)
    _check("fmsa_gptq_permute_rows",
           lib().fmsa_gptq_permute_rows(_ptr(qweight), _ptr(perm), K, N, _ptr(out), _stream(out)))
    return out


def permute_cols(x2d, perm, gather: bool):
    M, C = x2d.shape
    out = torch.empty((M, C), dtype=x2d.dtype, device=x2d.device)
    _check("fmsa_permute_cols",
           lib().fmsa_permute_cols(_ptr(x2d), x2d.stride(0), _ptr(perm), M, C, int(gather), act_enum(x2d.dtype),
                                   _ptr(out), out.stride(0), _stream(out)))
    return out


def lora_down(x2d, wd, out=None):
    """out [M, r] = x2d [M, C] @ wd [r, C]^T.  `out` may be a column slice of a wider buffer."""
    return (_native or native()).lora_down(x2d, wd, out)


LORA_DOWN_MAX_JOBS = 3
LORA_DOWN_BATCH_TOKENS = 2047  # from 2048 tokens on a product fills the chip by itself (and takes another kernel)


def lora_down_batch(jobs):
    """jobs: (x2d, wd, out or None) triples over the same M tokens; the list of lora_down(x2d, wd, out).  With few tokens
    one launch (and one of column sums) per LORA_DOWN_MAX_JOBS of them, single calls otherwise."""
    return (_native or native()).lora_down_batch(jobs, LORA_DOWN_BATCH_TOKENS)


def _workspace(nbytes: int, device) -> torch.Tensor:
    """Partial-sum buffer of one call.  A call is two launches, one writing the sums and one reading them, and another
    thread's call on the same stream may come between them; a captured graph keeps its address.  So no two calls share
    one: torch's allocator hands it out in stream order, or from the graph's own pool under capture."""
    return torch.empty(max(nbytes, 16), dtype=torch.uint8, device=device)


def lora_grad(L, R, scale: float, transpose_out: bool, out_dtype=torch.float32):
    """scale * L[M, r]^T @ R[M, C] -> [r, C] (or [C, r] when transpose_out)."""
    M, r = L.shape
    C = R.shape[1]
    assert R.shape[0] == M and L.stride(1) == 1 and R.stride(1) == 1 and L.dtype == R.dtype
    out = torch.empty((C, r) if transpose_out else (r, C), dtype=out_dtype, device=R.device)
    nbytes = lib().fmsa_lora_grad_workspace(M, C, r)
    ws = _workspace(nbytes, R.device)
    _check("fmsa_lora_grad",
           lib().fmsa_lora_grad(_ptr(L), L.stride(0), _ptr(R), R.stride(0), M, C, r, float(scale), int(transpose_out),
                                act_enum(R.dtype), _DTYPE_ENUM[out_dtype], _ptr(out), _ptr(ws), ws.numel(), _stream(out)))
    return out


LORA_GRAD_STATIC_BYTES = 16 << 20


def lora_grad_static(L, R, scale: float, transpose_out: bool, out):
    """lora_grad through the entry point that allocates nothing: the partial sums go to a buffer inside the
    library's device image (LORA_GRAD_STATIC_BYTES; larger requests raise), `out` is the caller's.  Calls that
    overlap on one GPU share that buffer and race."""
    M, r = L.shape
    C = R.shape[1]
    assert R.shape[0] == M and L.stride(1) == 1 and R.stride(1) == 1 and L.dtype == R.dtype
    assert out.is_contiguous() and tuple(out.shape) == ((C, r) if transpose_out else (r, C))
    assert L.device == R.device == out.device
    with torch.cuda.device(out.device):  # the library uses the buffer of the thread's current device
        _check("fmsa_lora_grad_static",
               lib().fmsa_lora_grad_static(_ptr(L), L.stride(0), _ptr(R), R.stride(0), M, C, r, float(scale), int(transpose_out),
                                           act_enum(R.dtype), _DTYPE_ENUM[out.dtype], _ptr(out), _stream(out)))
    return out


LORA_GRAD_MAX_JOBS = 8


LORA_GRAD_T_MAX_RANK = 32  # fmsa_lora_grad_batch computes T next to the gradient only up to this rank


def lora_grad_batch(jobs):
    """jobs: (L, R, scale, transpose_out, out_dtype[, Wt, T_out]) tuples over the same M tokens; returns
    the list of scale * L^T @ R, each as lora_grad would give it, from one launch of each pass per
    LORA_GRAD_MAX_JOBS jobs.  A job with Wt [r, C] and T_out [M, r] (may be a column slice) also gets
    T_out = R @ Wt^T from the same pass over R (all ranks of such a call <= LORA_GRAD_T_MAX_RANK)."""
    return (_native or native()).lora_grad_batch(jobs, LORA_GRAD_MAX_JOBS)


def gptq_lora_fwd(x2d, projs: Sequence[dict], mode: int = FWD_LINEAR, rope=None, split: bool = False):
    """projs: dicts with keys w (GptqWeight), U, B, bias (tensors or None), r, s.
    Returns the list of outputs Y_p [M, N_p]; in SWIGLU mode returns (e, g, h).
    rope = (cos2d, sin2d, head_dim, proj_mask): LINEAR mode only; the projections whose bit is set in proj_mask
    leave with the rotary embedding applied (token row m takes row m % cos2d.shape[0] of the tables).
    split=True lets the call cut tiles that do not fill the chip along K, and take the kernel for few tokens (other, still
    fixed, orders of the fp32 sums)."""
    if rope is None:
        return (_native or native()).gptq_lora_fwd(x2d, projs, mode, split)
    cos2d, sin2d, head_dim, proj_mask = rope
    assert mode == FWD_LINEAR and cos2d.shape == sin2d.shape and cos2d.dtype == sin2d.dtype
    assert cos2d.stride(1) == 1 and sin2d.stride(1) == 1 and cos2d.stride(0) == sin2d.stride(0) and cos2d.is_cuda
    if cos2d.dim() != 2 or cos2d.shape[1] < int(head_dim) // 2:
        raise ValueError("cos / sin must be [positions, >= head_dim / 2]")
    M = x2d.shape[0]
    arr = (FwdProj * len(projs))()
    outs = []
    for i, p in enumerate(projs):
        w = p["w"]
        y = x2d.new_empty((M, w.N))
        outs.append(y)
        U = p.get("U") if p["r"] else None
        assert U is None or U.stride(1) == 1
        arr[i] = FwdProj(w, _ptr(U), 0 if U is None else U.stride(0), _ptr(p.get("B")) if p["r"] else None,
                         _ptr(p.get("bias")), _ptr(y), y.stride(0), int(p["r"]), float(p["s"] or 0.0))
    desc = Rope(_ptr(cos2d), _ptr(sin2d), cos2d.stride(0), cos2d.shape[0], int(head_dim), _DTYPE_ENUM[cos2d.dtype], int(proj_mask))
    _check("fmsa_gptq_lora_fwd_rope",
           lib().fmsa_gptq_lora_fwd_rope(arr, len(projs), _ptr(x2d), x2d.stride(0), M, ctypes.byref(desc),
                                         act_enum(x2d.dtype), _stream(x2d)))
    return outs


FEW_TOKENS = 64  # up to here a pass without a graph goes straight from the adapters' parameters


def lora_few_ok(x2d, w: GptqWeight, A, B) -> bool:
    """Whether lora_few takes a projection (weight w, not act-order; adapter parameters A, B or None) as it is."""
    if x2d.shape[0] > FEW_TOKENS or w.group_size % 64:
        return False
    if A is None:
        return True
    r = A.shape[0]
    return (A.dtype == B.dtype and (A.dtype == torch.float32 or A.dtype == x2d.dtype) and A.is_cuda and B.is_cuda and r % 8 == 0
            and 0 < r <= 128 and A.is_contiguous() and B.is_contiguous() and (A.data_ptr() | B.data_ptr()) % 16 == 0)


def lora_few(x2d, projs, mode: int = FWD_LINEAR):
    """projs: (GptqWeight, A, B, bias, s) with the adapter's own parameters (None: no adapter).  The outputs of
    gptq_lora_fwd([...], split=True) on U = lora_down(x2d, A), to the last bit, from one launch for every U and one for every
    output; in SWIGLU mode h alone.  Nothing is kept for a backward.  None where gptq_lora_fwd would not take the kernel for
    few tokens."""
    return (_native or native()).lora_few(x2d, projs, mode)


def gptq_lora_fwd_splits(weights, M: int) -> bool:
    """Whether a LINEAR launch of these weights over M tokens, and a rotating pass over its outputs, is expected to be faster than
    the launch that rotates in its epilogue: its tiles are cut, or lower than the rotating ones and enough is won that way."""
    arr = (FwdProj * len(weights))()
    for i, w in enumerate(weights):
        arr[i].w = w
    return not lib().fmsa_gptq_lora_fwd_rope_pays(arr, len(weights), M)


def gptq_lora_bwd_dx(projs: Sequence[dict], M: int, K: int, mode: int = BWD_LINEAR, e=None, g=None, split: bool = False):
    """projs: dicts with keys w, nsz, dY, T, At, mask_src, r, s and optionally qweight_t, scale_f32, negzp_f16 (the
    weight's transposed twin and its tables, see gptq_transpose and gptq_negzp_f16).  LINEAR mode returns dX [M, K]; SWIGLU mode overwrites e <- d_g,
    g <- d_e and returns h.
    split=True lets a call on the twins cut tiles that do not fill the chip along the contraction (another, still fixed,
    order of the fp32 sums: the checkpoint layout's results, which run whole, then differ in their last bits)."""
    return (_native or native()).gptq_lora_bwd_dx(projs, M, K, mode, e, g, split)


def dx_twin_enabled() -> bool:
    """Whether prepared weights build the transposed twin the input-gradient kernel prefers (one more packed copy
    of every frozen weight, 4 bits per weight, plus fp32 scales).  FMSA_DX_TWIN=0 keeps the checkpoint layout only."""
    return os.environ.get("FMSA_DX_TWIN", "1") != "0"


def fwd_interleaved_enabled() -> bool:
    """Whether prepared weights build the interleaved copy the forward kernel's packed-half unpack reads for fp16
    activations (one more packed copy of every frozen weight, 4 bits per weight).  FMSA_FWD_INTERLEAVED=0 keeps the
    checkpoint layout only."""
    return os.environ.get("FMSA_FWD_INTERLEAVED", "1") != "0"


def gptq_negzp_f16(qzeros, N: int, zero_offset: int = 0):
    """fp16 [G, N] = -(1024 + zero point + zero_offset), exact in fp16: the offset table of the packed-half unpack
    (fmsa_bwd_proj.negzp_f16)."""
    shifts = torch.arange(0, 32, 4, device=qzeros.device, dtype=torch.int64)
    z = ((qzeros.to(torch.int64).unsqueeze(-1) >> shifts) & 0xF).reshape(qzeros.shape[0], -1)[:, :N]
    return (-(1024 + z + int(zero_offset))).to(torch.float16).contiguous()


def gptq_interleave(qweight):
    """The packed weight [K/8, N] with the nibbles of every word interleaved (element 2p at position p, element 2p + 1 at
    position 4 + p): what the forward kernel's packed-half unpack reads (GptqWeight.nibble_order = 1, fp16 activations)."""
    K8, N = qweight.shape
    assert qweight.dtype == torch.int32 and qweight.is_contiguous() and N % 4 == 0
    out = torch.empty_like(qweight)
    _check("fmsa_gptq_interleave", lib().fmsa_gptq_interleave(_ptr(qweight), K8 * 8, N, _ptr(out), _stream(qweight)))
    return out


def gptq_transpose(qweight):
    """The transposed twin [N/8, K] of a packed weight [K/8, N]: word [n8, k] holds q[k, 8 n8 + e], element 2p at nibble
    position p, element 2p + 1 at position 4 + p."""
    K8, N = qweight.shape
    assert qweight.dtype == torch.int32 and qweight.is_contiguous() and N % 8 == 0
    out = torch.empty((N // 8, K8 * 8), dtype=torch.int32, device=qweight.device)
    _check("fmsa_gptq_transpose", lib().fmsa_gptq_transpose(_ptr(qweight), K8 * 8, N, _ptr(out), _stream(qweight)))
    return out


def swiglu_fwd(e, g):
    """h = silu(e) * g with the reference's rounding points (standalone kernel)."""
    M, I = e.shape
    assert e.stride() == g.stride() and e.stride(1) == 1
    h = torch.empty_like(e)
    _check("fmsa_swiglu_fwd", lib().fmsa_swiglu_fwd(_ptr(e), _ptr(g), _ptr(h), M, I, e.stride(0), act_enum(e.dtype), _stream(e)))
    return h


def swiglu_bwd(dh, e, g):
    """In place: e <- d_g, g <- d_e; returns h."""
    M, I = e.shape
    assert e.stride() == g.stride() and e.stride(1) == 1 and dh.stride(1) == 1
    h = torch.empty_like(e)
    _check("fmsa_swiglu_bwd", lib().fmsa_swiglu_bwd(_ptr(dh), dh.stride(0), _ptr(e), _ptr(g), _ptr(h), M, I, e.stride(0),
                                                    act_enum(e.dtype), _stream(e)))
    return h


def nf4_dequant(packed, absmax_q, absmax2, code2, code, offset: float, shape, blocksize: int, blocksize2: int,
                out_dtype=torch.bfloat16):
    """Dense [N, K] weight of a bitsandbytes NF4 tensor with double-quantised absmax."""
    N, K = shape
    w = Nf4Weight(packed.data_ptr(), absmax_q.data_ptr(), absmax2.data_ptr(), code2.data_ptr(), code.data_ptr(),
                  float(offset), N, K, blocksize, blocksize2)
    out = torch.empty((N, K), dtype=out_dtype, device=packed.device)
    _check("fmsa_nf4_dequant", lib().fmsa_nf4_dequant(ctypes.byref(w), _DTYPE_ENUM[out_dtype], _ptr(out), _stream(out)))
    return out


def nf4_prepare(packed, absmax_q, absmax2, code2, offset: float, shape, blocksize: int, blocksize2: int):
    """(qweight int32 [K/8, N], block_scale fp32 [K / blocksize, N]) of an NF4 tensor [N, K]: the
    one-time re-layout the fused kernels read (see make_codebook_weight)."""
    N, K = shape
    w = Nf4Weight(packed.data_ptr(), absmax_q.data_ptr(), absmax2.data_ptr(), code2.data_ptr(), None, float(offset), N, K,
                  blocksize, blocksize2)
    qweight = torch.empty((K // 8, N), dtype=torch.int32, device=packed.device)
    block_scale = torch.empty((K // blocksize, N), dtype=torch.float32, device=packed.device)
    _check("fmsa_nf4_prepare", lib().fmsa_nf4_prepare(ctypes.byref(w), _ptr(qweight), _ptr(block_scale), _stream(qweight)))
    return qweight, block_scale


LORA_PACK_MAX_JOBS = 4


def lora_pack_batch(adapters, act_dtype):
    """adapters: (lora_A.weight [r, K], lora_B.weight [N, r], A16_out or None) triples (fp32 / bf16 / fp16
    parameters).  Returns one (A16 [r, K], At16 [K, r], B16 [N, r], Bt16 [r, N]) per adapter in `act_dtype`,
    from one launch per LORA_PACK_MAX_JOBS adapters.  `A16_out` (contiguous [r, K]) lets the caller place A16
    inside a larger stacked matrix."""
    return (_native or native()).lora_pack_batch(adapters, act_dtype, LORA_PACK_MAX_JOBS)


def lora_pack(A, B, act_dtype, A16_out=None):
    """lora_pack_batch for one adapter."""
    return lora_pack_batch([(A, B, A16_out)], act_dtype)[0]


def rms_layernorm_fwd(x2d, weight, eps: float, gemma: bool = False):
    """(Y [M, C] in x2d's dtype, r [M] fp32 = 1 / rms) of an RMS layer norm over the rows of x2d."""
    return (_native or native()).rms_layernorm_fwd(x2d, weight, eps, gemma)


def rms_layernorm_bwd(dy2d, x2d, weight, r, gemma: bool = False):
    """Overwrites dy2d with dX and returns it."""
    return (_native or native()).rms_layernorm_bwd(dy2d, x2d, weight, r, gemma)


def rope_embedding_(q2d, cos2d, sin2d, n_heads: int, head_dim: int, backward: bool = False, strided: bool = False):
    """In place on q2d [M, n_heads * head_dim]; row m uses row m % cos2d.shape[0] of cos / sin.  strided=True takes
    [batch, seq, n_heads, head_dim] of any strides instead and returns new rows (rope_embedding_strided)."""
    if strided:
        assert q2d.shape[2:] == (n_heads, head_dim)
        return rope_embedding_strided(q2d, cos2d, sin2d, backward)
    return (_native or native()).rope_embedding_(q2d, cos2d, sin2d, n_heads, head_dim, backward)


def rope_embedding_pair_(q2d, k2d, cos2d, sin2d, head_dim: int):
    """rope_embedding_ of q2d [M, n_heads * head_dim] and k2d [M, k_heads * head_dim], which do not overlap, in one launch."""
    return (_native or native()).rope_embedding_pair_(q2d, k2d, cos2d, sin2d, head_dim)


def rope_strided_ok(q4d, cos2d, sin2d) -> bool:
    """Whether rope_embedding_strided takes q4d [batch, seq, heads, head_dim] as it lies in memory."""
    esz, csz = q4d.element_size(), cos2d.element_size()
    return (q4d.is_cuda and q4d.numel() > 0 and q4d.dtype in _DTYPE_ENUM and q4d.stride(3) == 1 and q4d.shape[3] % 16 == 0
            and q4d.data_ptr() % 16 == 0 and all(q4d.stride(i) >= 0 and q4d.stride(i) * esz % 16 == 0 for i in range(3))
            and cos2d.data_ptr() % 16 == 0 and sin2d.data_ptr() % 16 == 0 and cos2d.stride(0) * csz % 16 == 0)


def rope_embedding_strided(q4d, cos2d, sin2d, backward: bool = False):
    """The rotation of q4d [batch, seq, heads, head_dim], any strides (see rope_strided_ok), as contiguous rows
    [batch * seq, heads * head_dim]; row m uses row m % cos2d.shape[0] of cos / sin.  q4d is left alone."""
    return (_native or native()).rope_embedding_strided(q4d, cos2d, sin2d, backward)


def cross_entropy_fwd(logits2d, labels):
    """(losses [M] fp32, logsumexp [M] fp32); labels int64 [M], -100 ignored."""
    if not (logits2d.is_cuda and labels.is_cuda):
        raise RuntimeError("fmsa_hip needs GPU tensors")
    M, V = logits2d.shape
    assert logits2d.stride(1) == 1 and labels.dtype == torch.int64 and labels.is_contiguous() and labels.numel() == M
    losses = torch.empty(M, dtype=torch.float32, device=logits2d.device)
    lse = torch.empty(M, dtype=torch.float32, device=logits2d.device)
    _check("fmsa_cross_entropy_fwd", lib().fmsa_cross_entropy_fwd(_ptr(logits2d), logits2d.stride(0), _ptr(labels), M, V,
                                                                  _DTYPE_ENUM[logits2d.dtype], _ptr(losses), _ptr(lse), _stream(logits2d)))
    return losses, lse


def cross_entropy_bwd_(logits2d, dlosses, lse, labels):
    """Overwrites logits2d with the gradient and returns it; dlosses [M] fp32 (any stride, 0 included)."""
    M, V = logits2d.shape
    assert dlosses.dtype == torch.float32 and dlosses.numel() == M and dlosses.dim() == 1
    _check("fmsa_cross_entropy_bwd", lib().fmsa_cross_entropy_bwd(_ptr(logits2d), logits2d.stride(0), _ptr(dlosses), dlosses.stride(0),
                                                                  _ptr(lse), _ptr(labels), M, V, _DTYPE_ENUM[logits2d.dtype],
                                                                  _stream(logits2d)))
    return logits2d


def cross_entropy_rows_fwd(logits3d, labels, seq_out: int):
    """(losses, logsumexp), fp32 [n_seq * seq_out], of rows 0 .. seq_out - 1 of every sequence of contiguous 16-bit logits
    [n_seq, seq_in, V]; labels int64 [n_seq * seq_out], -100 ignored.  For callers that want them by rows: the loss operator
    takes causal_lm_loss_fwd, which sums them on the way."""
    n_seq, seq_in, V = logits3d.shape
    rows = n_seq * seq_out
    assert logits3d.is_contiguous() and labels.dtype == torch.int64 and labels.is_contiguous() and labels.numel() == rows
    losses = torch.empty(rows, dtype=torch.float32, device=logits3d.device)
    lse = torch.empty(rows, dtype=torch.float32, device=logits3d.device)
    _check("fmsa_cross_entropy_rows_fwd",
           lib().fmsa_cross_entropy_rows_fwd(_ptr(logits3d), V, _ptr(labels), n_seq, seq_in, seq_out, V, act_enum(logits3d.dtype),
                                             _ptr(losses), _ptr(lse), _stream(logits3d)))
    return losses, lse


def cross_entropy_rows_bwd(logits3d, dlosses, lse, labels, seq_out: int):
    """Gradient of cross_entropy_rows_fwd's losses, a tensor of its own; dlosses fp32 (any stride, 0 included)."""
    n_seq, seq_in, V = logits3d.shape
    assert dlosses.dtype == torch.float32 and dlosses.dim() == 1 and dlosses.numel() == n_seq * seq_out
    grad = torch.empty_like(logits3d)
    _check("fmsa_cross_entropy_rows_bwd",
           lib().fmsa_cross_entropy_rows_bwd(_ptr(logits3d), _ptr(grad), V, _ptr(dlosses), dlosses.stride(0), _ptr(lse), _ptr(labels),
                                             n_seq, seq_in, seq_out, V, act_enum(logits3d.dtype), _stream(logits3d)))
    return grad


def causal_lm_loss_fwd(logits3d, labels, label_stride: int, seq_out: int, mean: bool, keep: bool):
    """(loss, saved): the sum (mean: over the labels that are not -100) of cross_entropy_rows_fwd's losses of contiguous 16-bit
    logits [n_seq, seq_in, V], a scalar; label of row t of sequence q: element q * label_stride + t of the int64 `labels`.
    saved, with keep: what causal_lm_loss_bwd takes, none of it the caller's (the rows with a label are copied, so that the
    logits may be overwritten before the backward)."""
    n_seq, seq_in, V = logits3d.shape
    rows, dev = n_seq * seq_out, logits3d.device
    assert logits3d.is_contiguous() and labels.dtype == torch.int64 and labels.is_cuda
    loss = torch.empty((), dtype=torch.float32, device=dev)
    count = torch.empty((), dtype=torch.float32, device=dev)
    lse = torch.empty(rows, dtype=torch.float32, device=dev)
    targets = kept = None
    if keep:
        targets = torch.empty(rows, dtype=torch.int64, device=dev)
        offset = logits3d.data_ptr() % 16 // logits3d.element_size()  # a row begins where it does in the logits, modulo 16 bytes
        kept = logits3d.new_empty(offset + logits3d.numel())[offset:].view(logits3d.shape)
    nbytes = lib().fmsa_causal_lm_loss_workspace(n_seq, seq_out, V)
    ws = _workspace(nbytes, dev)
    _check("fmsa_causal_lm_loss_fwd",
           lib().fmsa_causal_lm_loss_fwd(_ptr(logits3d), _ptr(kept), V, _ptr(labels), int(label_stride), n_seq, seq_in, seq_out, V,
                                         act_enum(logits3d.dtype), int(mean), _ptr(loss), _ptr(count), _ptr(lse), _ptr(targets), _ptr(ws),
                                         ws.numel(), _stream(logits3d)))
    return loss, (kept, lse, targets, count) if keep else None


def causal_lm_loss_bwd(kept, lse, targets, count, dloss, seq_out: int):
    """Gradient of causal_lm_loss_fwd's logits, a tensor of its own; dloss an fp32 scalar on the GPU."""
    n_seq, seq_in, V = kept.shape
    assert dloss.dtype == torch.float32 and dloss.numel() == 1 and dloss.is_cuda
    grad = torch.empty_like(kept)
    _check("fmsa_causal_lm_loss_bwd",
           lib().fmsa_causal_lm_loss_bwd(_ptr(kept), _ptr(grad), V, _ptr(dloss), _ptr(count), _ptr(lse), _ptr(targets), n_seq, seq_in, seq_out,
                                         V, act_enum(kept.dtype), _stream(kept)))
    return grad


def cross_entropy_fused_(logits2d, labels, scale=None, label_smoothing=0.0, ignore_index=-100, losses_out=None):
    """Overwrites logits2d with scale * d(loss)/d(logits) and returns (losses [M] fp32, already scaled;
    logits2d).  `scale` is a 1-element fp32 GPU tensor (None = 1)."""
    if not (logits2d.is_cuda and labels.is_cuda):
        raise RuntimeError("fmsa_hip needs GPU tensors")
    M, V = logits2d.shape
    assert logits2d.stride(1) == 1 and labels.dtype == torch.int64 and labels.is_contiguous() and labels.numel() == M
    assert scale is None or (scale.is_cuda and scale.dtype == torch.float32 and scale.numel() == 1)
    losses = losses_out if losses_out is not None else torch.empty(M, dtype=torch.float32, device=logits2d.device)
    assert losses.dtype == torch.float32 and losses.is_contiguous() and losses.numel() == M
    _check("fmsa_cross_entropy_fused",
           lib().fmsa_cross_entropy_fused(_ptr(logits2d), logits2d.stride(0), _ptr(labels), M, V, _DTYPE_ENUM[logits2d.dtype],
                                          int(ignore_index), _ptr(scale) if scale is not None else None, float(label_smoothing),
                                          _ptr(losses), _stream(logits2d)))
    return losses, logits2d
