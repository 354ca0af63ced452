"""PyTorch-ROCm custom operators ``torch.ops.sgl_kernel.*`` backed by the gfx950 C ABI.

The operator names and schema strings are the reference's own
(sgl-kernel/csrc/common_extension.cc:158-181); the implementations are native
(``csrc/torch_binding.cpp``, the extension module ``sglang_amd._native``) and registered for the
``CUDA`` dispatch key, which is the HIP device under PyTorch-ROCm.  Each checks its arguments
the way the reference's host function does (same conditions, same wording, RuntimeError),
allocates outputs and workspaces through torch's caching allocator (so nothing here breaks HIP
graph capture) and passes raw device pointers plus the current stream to
``libmi355_qlinear.so``.  The functions below are the same calls without the dispatcher, with
their Python signatures.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import _lib
from ._lib import check, lib

lib()  # fail now, loudly, if the native library is missing
try:
    from . import _native
except ImportError as e:
    raise ImportError(f"sglang_amd._native cannot be loaded: build it with `make -C {_lib._CSRC}` (or __graft_entry__.build()). "
                      "The quantized-linear operators have no other host path.") from e

_native.set_error_class(_lib.Mi355Error)

_DT = {
    torch.float32: _lib.F32,
    torch.float16: _lib.F16,
    torch.bfloat16: _lib.BF16,
    torch.float8_e4m3fn: _lib.FP8_E4M3FN,
    torch.int8: _lib.I8,
    torch.int32: _lib.I32,
}

SCHEMAS = {
    "int8_scaled_mm": "int8_scaled_mm(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, "
    "ScalarType out_dtype, Tensor? bias) -> Tensor",
    "fp8_blockwise_scaled_mm": "fp8_blockwise_scaled_mm(Tensor mat_a, Tensor mat_b, Tensor scales_a, "
    "Tensor scales_b, ScalarType out_dtype) -> Tensor",
    "sgl_per_token_group_quant_8bit": "sgl_per_token_group_quant_8bit(Tensor input, Tensor output_q, "
    "Tensor output_s, int group_size, float eps, float fp8_min, float fp8_max, bool scale_ue8m0) -> ()",
    "sgl_per_token_group_quant_8bit_v2": "sgl_per_token_group_quant_8bit_v2(Tensor input, Tensor output_q, "
    "Tensor output_s, int group_size, float eps, float fp8_min, float fp8_max, bool scale_ue8m0, "
    "bool fuse_silu_and_mul, Tensor? masked_m) -> ()",
    "fp8_scaled_mm": "fp8_scaled_mm(Tensor mat_a, Tensor mat_b, Tensor scales_a, Tensor scales_b, ScalarType out_dtype, "
    "Tensor? bias) -> Tensor",
    "sgl_per_token_quant_fp8": "sgl_per_token_quant_fp8(Tensor input, Tensor output_q, Tensor output_s) -> ()",
    "sgl_per_tensor_quant_fp8": "sgl_per_tensor_quant_fp8(Tensor input, Tensor output_q, Tensor output_s, bool is_static) -> ()",
    "fp8_blockwise_scaled_grouped_mm": "fp8_blockwise_scaled_grouped_mm(Tensor output, Tensor a_ptrs, Tensor b_ptrs, "
    "Tensor out_ptrs, Tensor a_scales_ptrs, Tensor b_scales_ptrs, Tensor a, Tensor b, Tensor scales_a, Tensor scales_b, "
    "Tensor stride_a, Tensor stride_b, Tensor stride_c, Tensor layout_sfa, Tensor layout_sfb, Tensor problem_sizes, "
    "Tensor expert_offsets, Tensor workspace) -> ()",
    "es_fp8_blockwise_scaled_grouped_mm": "es_fp8_blockwise_scaled_grouped_mm(Tensor output, Tensor a, Tensor b, Tensor scales_a, "
    "Tensor scales_b, Tensor stride_a, Tensor stride_b, Tensor stride_d, Tensor problem_sizes, Tensor expert_offsets, "
    "Tensor workspace) -> ()",
}


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _require(cond: bool, msg: str) -> None:
    if not cond:
        raise RuntimeError(msg)


# ---------------------------------------------------------------- quantizers

def sgl_per_token_group_quant_8bit(input, output_q, output_s, group_size, eps, fp8_min, fp8_max, scale_ue8m0):
    """sgl-kernel/csrc/gemm/per_token_group_quant_8bit.cu:116-217: q = x / (amax / max)."""
    _native.sgl_per_token_group_quant_8bit(input, output_q, output_s, group_size, eps, fp8_min, fp8_max, scale_ue8m0)


def sgl_per_token_group_quant_8bit_v2(input, output_q, output_s, group_size, eps, fp8_min, fp8_max, scale_ue8m0,
                                      fuse_silu_and_mul, masked_m):
    """sgl-kernel/csrc/gemm/per_token_group_quant_8bit_v2.cu:394-514: q = x * (max / amax)."""
    _native.sgl_per_token_group_quant_8bit_v2(input, output_q, output_s, group_size, eps, fp8_min, fp8_max, scale_ue8m0,
                                              fuse_silu_and_mul, masked_m)


def sgl_per_token_quant_fp8(input, output_q, output_s):
    """sgl-kernel/csrc/gemm/per_token_quant_fp8.cu:162-227."""
    _native.sgl_per_token_quant_fp8(input, output_q, output_s)


def block_cast_to_fp8(x: torch.Tensor):
    """x [m, n] -> (e4m3fn [m, n], fp32 power-of-two scales [ceil(m/128), ceil(n/128)]): per_block_cast_to_fp8 of
    python/sglang/srt/layers/quantization/fp8_utils.py:487-500 as one kernel."""
    _require(x.is_cuda and x.dim() == 2, "block_cast_to_fp8: a 2-D CUDA tensor is expected")
    _require(x.dtype in (torch.float32, torch.float16, torch.bfloat16), "block_cast_to_fp8: unsupported dtype")
    x = x.contiguous()
    m, n = x.shape
    q = torch.empty((m, n), dtype=torch.float8_e4m3fn, device=x.device)
    s = torch.empty(((m + 127) // 128, (n + 127) // 128), dtype=torch.float32, device=x.device)
    check(lib().mi355_block_cast_to_fp8(x.data_ptr(), _DT[x.dtype], q.data_ptr(), s.data_ptr(), m, n, _stream()))
    return q, s


def block_dequant_fp8(q: torch.Tensor, s: torch.Tensor, dtype: torch.dtype):
    """q [n, k] e4m3fn, s [ceil(n/128), ceil(k/128)] -> [n, k] of `dtype`: block_quant_dequant (fp8_utils.py:392-413)."""
    _require(q.is_cuda and q.dim() == 2 and q.dtype == torch.float8_e4m3fn, "block_dequant_fp8: a 2-D e4m3fn CUDA tensor is expected")
    n, k = q.shape
    _require(tuple(s.shape) == ((n + 127) // 128, (k + 127) // 128), "block_dequant_fp8: scale shape mismatch")
    _require(dtype in (torch.float32, torch.float16, torch.bfloat16), "block_dequant_fp8: unsupported dtype")
    q = q.contiguous()
    s = s.to(torch.float32).contiguous()
    out = torch.empty((n, k), dtype=dtype, device=q.device)
    check(lib().mi355_block_dequant_fp8(q.data_ptr(), s.data_ptr(), out.data_ptr(), _DT[dtype], n, k, _stream()))
    return out


def sgl_per_tensor_quant_fp8(input, output_q, output_s, is_static):
    """sgl-kernel/csrc/gemm/per_tensor_quant_fp8.cu:102-130.  Dynamic mode merges block maxima into `output_s` with an
    atomic max, so the caller passes zeros (the reference's scaled_fp8_quant does)."""
    _native.sgl_per_tensor_quant_fp8(input, output_q, output_s, is_static)


def static_quant_fp8_repeat(input, output_q, scale, scale_rows):
    """Static per-tensor quantization that also writes the scale once per row (static_quant_fp8 with repeat_scale,
    python/sglang/srt/layers/quantization/fp8_kernel.py:635-665)."""
    _native.static_quant_fp8_repeat(input, output_q, scale, scale_rows)


def per_token_quant_int8(x2d: torch.Tensor, q: torch.Tensor, s: torch.Tensor, x_sum: Optional[torch.Tensor] = None) -> None:
    """Codes and scales of the rows of `x2d`; with `x_sum` ([M], the input's type) also the row sums."""
    _native.per_token_quant_int8(x2d, q, s, x_sum)


# ---------------------------------------------------------------- GEMMs

def fp8_blockwise_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype):
    """sgl-kernel/csrc/gemm/fp8_blockwise_gemm_kernel.cu:368-465."""
    return _native.fp8_blockwise_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype)


def block_fp8_matmul(A2d, B, As2d, Bs, out2d):
    """The ``w8a8_block_fp8_matmul`` contract on flattened operands: B [N, K] row-major weight,
    Bs [ceil(N/128), ceil(K/128)], As2d [M, ceil(K/128)] any strides, ragged N and K allowed."""
    _native.block_fp8_matmul(A2d, B, As2d, Bs, out2d)
    return out2d


def fp8_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias: Optional[torch.Tensor] = None):
    """sgl-kernel/csrc/gemm/fp8_gemm_kernel.cu:1450-1532."""
    return _native.fp8_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias)


def int8_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias: Optional[torch.Tensor] = None):
    """sgl-kernel/csrc/gemm/int8_gemm_kernel.cu:663-747."""
    return _native.int8_scaled_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias)


def int8_mm_raw_accumulators(mat_a: torch.Tensor, mat_b: torch.Tensor) -> torch.Tensor:
    """int32 accumulators of ``int8_scaled_mm`` before its epilogue (same kernel, epilogue skipped)."""
    return _native.int8_mm_raw_accumulators(mat_a, mat_b)


def fp8_blockwise_mm_ue8m0(a: torch.Tensor, b: torch.Tensor, a_words: torch.Tensor, b_words: torch.Tensor,
                           out_dtype: torch.dtype, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Blockwise FP8 GEMM with packed power-of-two scales on both sides: a [M, K] e4m3fn, b [N, K] e4m3fn (the weight as
    stored), a_words int32 [M, ceil(K/512)] and b_words int32 [N, ceil(K/512)], both with stride 1 along their first
    dimension (the layouts of create_per_token_group_quant_fp8_output_scale(scale_ue8m0=True) and
    fp8_utils.transform_scale_ue8m0).  What deep_gemm's gemm_nt_f8f8bf16 computes for the reference
    (python/sglang/srt/layers/quantization/fp8_kernel.py:1047-1065)."""
    return _native.fp8_blockwise_mm_ue8m0(a, b, a_words, b_words, out_dtype, bias)


# ---------------------------------------------------------------- one-call linears

def block_fp8_linear_ue8m0(x2d: torch.Tensor, weight: torch.Tensor, weight_words: torch.Tensor, bias: Optional[torch.Tensor],
                           out_dtype: torch.dtype) -> torch.Tensor:
    """One block-FP8 linear layer with packed power-of-two scales in one C-ABI call: x2d [M, K] (contiguous bf16/fp16,
    K % 128 == 0) is quantized per 1 x 128 group with UE8M0 scales into the workspace and multiplied with `weight` [N, K]
    e4m3fn, whose packed scale words are `weight_words` int32 [N, ceil(K/512)] (fp8_utils.transform_scale_ue8m0).  The
    result is that of the quantizer call of deepgemm_w8a8_block_fp8_linear_with_fallback followed by
    `fp8_blockwise_mm_ue8m0`, bit for bit."""
    return _native.block_fp8_linear_ue8m0(x2d, weight, weight_words, bias, out_dtype)


def fp8_per_token_linear(x2d: torch.Tensor, weight_kn: torch.Tensor, weight_scale: torch.Tensor, bias: Optional[torch.Tensor],
                         out_dtype: torch.dtype) -> torch.Tensor:
    """One per-token x per-channel FP8 linear layer in one C-ABI call: per-token quantization of x2d [M, K] (contiguous
    bf16/fp16/fp32) into the workspace, then the GEMM with `weight_kn` [K, N] e4m3fn column-major, per-channel `weight_scale`
    ([N] fp32) and bias in its epilogue.  The result is that of `sgl_per_token_quant_fp8` followed by `fp8_scaled_mm`, bit
    for bit."""
    return _native.fp8_per_token_linear(x2d, weight_kn, weight_scale, bias, out_dtype)


def block_fp8_linear(x2d: torch.Tensor, weight: torch.Tensor, weight_scale: torch.Tensor,
                     bias: Optional[torch.Tensor], out_dtype: torch.dtype, by_reciprocal: bool = False) -> torch.Tensor:
    """One block-FP8 linear layer (1x128 activation groups, 128x128 weight blocks) in one C-ABI call: the activation is
    quantized into the workspace, multiplied, and the bias is added in the GEMM epilogue.  x2d [M, K] contiguous
    bf16/fp16/fp32 with K % 128 == 0, weight [N, K] e4m3fn, weight_scale [ceil(N/128), K/128] (any strides).
    by_reciprocal: the quantizer computes q = x * (1 / s) (the reference's row-major-scale path, fp8_kernel.py:156-158)
    instead of q = x / s (its M-major-scale path)."""
    return _native.block_fp8_linear(x2d, weight, weight_scale, bias, out_dtype, by_reciprocal)


def int8_linear(x2d: torch.Tensor, weight_kn: torch.Tensor, weight_scale: torch.Tensor, bias: Optional[torch.Tensor],
                out_dtype: torch.dtype) -> torch.Tensor:
    """One INT8 linear layer in one C-ABI call: per-token quantization of x2d [M, K] (contiguous bf16/fp16/fp32) into the
    workspace, then the INT8 GEMM with `weight_kn` [K, N] int8 column-major, per-channel `weight_scale` ([N] fp32) and bias in
    its epilogue.  The result is that of `per_token_quant_int8` followed by `int8_scaled_mm`, bit for bit."""
    return _native.int8_linear(x2d, weight_kn, weight_scale, bias, out_dtype)


# ---------------------------------------------------------------- grouped FP8 GEMM (mixture-of-experts)

def fp8_blockwise_scaled_grouped_mm(output, a_ptrs, b_ptrs, out_ptrs, a_scales_ptrs, b_scales_ptrs, a, b, scales_a, scales_b,
                                    stride_a, stride_b, stride_c, layout_sfa, layout_sfb, problem_sizes, expert_offsets,
                                    workspace):
    """sgl-kernel/csrc/moe/fp8_blockwise_moe_kernel.cu:650-810 (checks :668-706).  ``a`` [total_m, K] e4m3fn row-major,
    ``b`` [E, K, N] e4m3fn column-major per expert (storage [E, N, K]), ``scales_a`` fp32 [total_m, K/128], ``scales_b``
    fp32 [E, K/128, N/128] (storage [E, N/128, K/128]), ``problem_sizes`` int32 [E, 3] and ``expert_offsets`` int32 [E] on
    the device, ``output`` [total_m, N] written in place.  The pointer, stride and scale-layout tensors are scratch of the
    reference's kernels: they are type-checked like there and not used.  ``workspace`` is used when it is large enough
    (the reference's callers pass hundreds of megabytes), otherwise a temporary one is allocated."""
    _native.fp8_blockwise_scaled_grouped_mm(
        output, a_ptrs, b_ptrs, out_ptrs, a_scales_ptrs, b_scales_ptrs, a, b, scales_a, scales_b, stride_a, stride_b, stride_c,
        layout_sfa, layout_sfb, problem_sizes, expert_offsets, workspace)


def es_fp8_blockwise_scaled_grouped_mm(output, a, b, scales_a, scales_b, stride_a, stride_b, stride_d, problem_sizes,
                                       expert_offsets, workspace):
    """sgl-kernel/csrc/expert_specialization/es_fp8_blockwise.cu:33-170: the same computation on the same layouts without
    the caller-provided scratch tensors.  The reference sorts experts into low / middle / high row counts and runs one
    tile configuration on each; here the device-built schedule does that per tile (256-row tiles and a small-tile rest)."""
    _native.es_fp8_blockwise_scaled_grouped_mm(output, a, b, scales_a, scales_b, stride_a, stride_b, stride_d, problem_sizes,
                                               expert_offsets, workspace)


# ---------------------------------------------------------------- registration

_registered = False
_torch_lib = None


def register() -> None:
    """Define the ``sgl_kernel`` operators (unless an installed sgl_kernel already did) and attach their
    fake implementations; the gfx950 ones are attached to the CUDA (= HIP) dispatch key by
    the extension module.  Idempotent."""
    global _registered, _torch_lib
    if _registered:
        return
    _torch_lib = torch.library.Library("sgl_kernel", "FRAGMENT")
    for name, schema in SCHEMAS.items():
        if not hasattr(torch.ops.sgl_kernel, name):
            _torch_lib.define(schema)

    def _fake_mm(mat_a, mat_b, scales_a, scales_b, out_dtype, bias=None):
        return mat_a.new_empty((mat_a.size(0), mat_b.size(1)), dtype=out_dtype)

    torch.library.register_fake("sgl_kernel::int8_scaled_mm", _fake_mm, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::fp8_blockwise_scaled_mm", _fake_mm, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::fp8_scaled_mm", _fake_mm, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::sgl_per_token_quant_fp8", lambda *a: None, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::sgl_per_tensor_quant_fp8", lambda *a: None, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::fp8_blockwise_scaled_grouped_mm", lambda *a: None, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::es_fp8_blockwise_scaled_grouped_mm", lambda *a: None, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::sgl_per_token_group_quant_8bit", lambda *a: None, lib=_torch_lib)
    torch.library.register_fake("sgl_kernel::sgl_per_token_group_quant_8bit_v2", lambda *a: None, lib=_torch_lib)
    _registered = True
