"""Forward passes of the FP8 linear methods on the gfx950 kernels.

The reference builds a block-FP8 linear out of three Python-level steps - quantize the activation per 1x128 group,
run the blockwise GEMM, `output += bias` on the already rounded output
(python/sglang/srt/layers/quantization/fp8_utils.py:184-214 for the CUTLASS path, :281-301 for the Triton path, chosen
by :139-149) - and a per-token x per-channel linear out of `sgl_per_token_quant_fp8` + `fp8_scaled_mm` (:565-853).
The two block-FP8 wrappers are different computations and are kept different here:

* `cutlass_w8a8_block_fp8_linear_with_fallback`: `q = x / s` codes with M-major scales, `fp8_blockwise_scaled_mm`,
  falling back to the Triton wrapper when N or K is not a multiple of 128;
* `triton_w8a8_block_fp8_linear`: `q = x * (1 / s)` codes with row-major scales, `w8a8_block_fp8_matmul`;

both add the bias to the rounded 16-bit output (a second rounding), as the reference does.
The linear methods first offer their operands to a native fast path (`_native.try_*`: the whole forward pass in one call for
plain contiguous 16-bit activations and the weight layouts of a loaded checkpoint, about 4 us of host time); it declines
anything else, among it every call that somebody looks at through PyTorch's dispatcher (dispatch and function modes, tracing,
vmap), and the Python below computes it, or raises.  Under `torch.compile` and export it is not asked: its tracer cannot
follow a C function.
`fused_w8a8_block_fp8_linear` is this library's own one-call variant (`mi355_fp8_block_linear`: codes and scales live
only in the call's workspace, bias added in fp32 before the single rounding); it is an opt-in, not what the reference's
names resolve to, because its outputs may differ from theirs in the last bit when a bias is present.
"""
from __future__ import annotations

import functools
from typing import Callable, List, Optional

import torch
from torch.compiler import is_dynamo_compiling

from . import _lib, _native, ops
from .fp8_kernel import (
    per_token_group_quant_fp8,
    scaled_fp8_quant,
    sglang_per_token_quant_fp8,
    static_quant_fp8,
    w8a8_block_fp8_matmul,
    w8a8_block_fp8_matmul_deepgemm,
    w8a8_block_fp8_matmul_triton,
)
from .sgl_kernel import fp8_blockwise_scaled_mm, fp8_scaled_mm


@functools.lru_cache(maxsize=4096)
def _one_call_takes_the_same_gemm(M: int, N: int, K: int) -> bool:
    """Whether the one-call linear multiplies with the kernel and tiling the GEMM entry point alone would take for this
    shape: then both add the same products in the same order and their results are the same bit for bit.  At some decode
    shapes the one-call linear takes another kernel (one that quantizes the tokens itself and is faster than a quantizer
    launch plus the GEMM entry point's choice); there the results agree to rounding, not bit for bit."""
    one = _lib.block_linear_plan(M, N, K)
    one.pop("quantizer")
    return one == _lib.gemm_plan("fp8", M, N, K)


def _quantize_and_multiply(input_2d: torch.Tensor, weight: torch.Tensor, block_size: List[int], weight_scale: torch.Tensor,
                           by_reciprocal: bool) -> Optional[torch.Tensor]:
    """The quantizer and the blockwise GEMM of a linear wrapper as one C-ABI call, where that call's preconditions hold
    (None otherwise, and the wrapper makes its two calls).  Codes and scales are those of the wrapper's quantizer, bit for
    bit; at decode sizes the GEMM kernel quantizes the tokens itself and there is no quantizer launch.  The product is the
    two calls' bit for bit wherever `_one_call_takes_the_same_gemm`, and within the GEMM's tolerance elsewhere (another
    kernel adds the same products in another order)."""
    ok = (list(block_size) == [128, 128] and input_2d.dtype in (torch.bfloat16, torch.float16) and input_2d.is_cuda
          and input_2d.is_contiguous() and input_2d.shape[0] > 0 and input_2d.shape[1] % 128 == 0 and weight.dim() == 2
          and weight.is_contiguous() and weight.dtype == torch.float8_e4m3fn and weight.shape[1] == input_2d.shape[1]
          and weight_scale.dtype == torch.float32
          and tuple(weight_scale.shape) == ((weight.shape[0] + 127) // 128, weight.shape[1] // 128))
    if not ok:
        return None
    return ops.block_fp8_linear(input_2d, weight, weight_scale, None, input_2d.dtype, by_reciprocal=by_reciprocal)


def triton_w8a8_block_fp8_linear(
    input: torch.Tensor,
    weight: torch.Tensor,
    block_size: List[int],
    weight_scale: torch.Tensor,
    input_scale: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """fp8_utils.py:281-301: row-major-scale quantizer (`x * (1 / s)`), the ragged-shape matmul, bias on the rounded output."""
    assert input_scale is None
    if not is_dynamo_compiling():
        output = _native.try_block_linear(input, weight, block_size, weight_scale, bias, True)
        if output is not None:
            return output
    input_2d = input.view(-1, input.shape[-1])
    output_shape = [*input.shape[:-1], weight.shape[0]]

    output = _quantize_and_multiply(input_2d, weight, block_size, weight_scale, by_reciprocal=True)
    if output is None:
        q_input, x_scale = per_token_group_quant_fp8(input_2d, block_size[1], column_major_scales=False)
        output = w8a8_block_fp8_matmul_triton(q_input, weight, x_scale, weight_scale, block_size, output_dtype=input_2d.dtype)
    if bias is not None:
        output += bias
    return output.to(dtype=input_2d.dtype).view(*output_shape)


def cutlass_w8a8_block_fp8_linear_with_fallback(
    input: torch.Tensor,
    weight: torch.Tensor,
    block_size: List[int],
    weight_scale: torch.Tensor,
    input_scale: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """fp8_utils.py:184-214: M-major-scale quantizer (`x / s`), `fp8_blockwise_scaled_mm` on the transposed views, bias on
    the rounded output; shapes with N or K not a multiple of 128 go to the Triton wrapper."""
    assert input_scale is None
    if not is_dynamo_compiling():
        output = _native.try_block_linear(input, weight, block_size, weight_scale, bias, False)
        if output is not None:
            return output

    shape_supported = weight.shape[0] % 128 == 0 and weight.shape[1] % 128 == 0
    if not shape_supported:
        return triton_w8a8_block_fp8_linear(input, weight, block_size, weight_scale, input_scale, bias)

    input_2d = input.view(-1, input.shape[-1])
    output_shape = [*input.shape[:-1], weight.shape[0]]

    output = _quantize_and_multiply(input_2d, weight, block_size, weight_scale, by_reciprocal=False)
    if output is None:
        q_input, x_scale = per_token_group_quant_fp8(input_2d, block_size[1], column_major_scales=True)
        output = fp8_blockwise_scaled_mm(q_input, weight.T, x_scale, weight_scale.T, out_dtype=input_2d.dtype)
    if bias is not None:
        output += bias
    return output.to(dtype=input_2d.dtype).view(*output_shape)


def dispatch_w8a8_block_fp8_linear() -> Callable:
    """fp8_utils.py:139-149 with the CUTLASS-class kernel available, which is the case on gfx950 with this library."""
    return cutlass_w8a8_block_fp8_linear_with_fallback


# the name `Fp8LinearMethod.apply` calls after dispatch
w8a8_block_fp8_linear = cutlass_w8a8_block_fp8_linear_with_fallback


def fused_w8a8_block_fp8_linear(
    input: torch.Tensor,
    weight: torch.Tensor,
    block_size: List[int],
    weight_scale: torch.Tensor,
    input_scale: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """This library's one-call block-FP8 linear (no counterpart in the reference): `x / s` codes and M-major scales
    written to the call's workspace (at decode sizes quantized inside the GEMM kernel), GEMM, bias added in fp32 in the
    GEMM epilogue and rounded once.  Without a bias its output equals `cutlass_w8a8_block_fp8_linear_with_fallback`'s bit
    for bit; with one it differs by at most the wrapper's extra rounding of the product (one rounding instead of two).  Needs K % 128 == 0 and
    a 16-bit input type."""
    assert input_scale is None
    if list(block_size) != [128, 128]:
        raise NotImplementedError("only 128x128 weight blocks with 1x128 activation groups are built")
    K = input.shape[-1]
    N = weight.shape[0]
    if K % 128 != 0 or input.dtype not in (torch.bfloat16, torch.float16):
        raise NotImplementedError("the one-call linear needs K % 128 == 0 and bf16/fp16 activations")
    x2d = input.reshape(-1, K)
    if not x2d.is_contiguous():
        x2d = x2d.contiguous()
    fused_bias = bias if bias is None or (bias.dtype == input.dtype and bias.is_contiguous()) else bias.to(input.dtype).contiguous()
    out = ops.block_fp8_linear(x2d, weight, weight_scale, fused_bias, input.dtype)
    return out.view(*input.shape[:-1], N)


def deepgemm_w8a8_block_fp8_linear_with_fallback(
    input: torch.Tensor,
    weight: torch.Tensor,
    block_size: List[int],
    weight_scale: torch.Tensor,
    input_scale: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
) -> torch.Tensor:
    """fp8_utils.py:217-255: the block-FP8 linear for checkpoints re-quantized to power-of-two scales
    (requant_weight_ue8m0): activations quantized with packed UE8M0 scales, the GEMM with the scales applied by the
    matrix instruction, bias added to the rounded output.  ``weight_scale`` is the packed int32 [N, ceil(K/512)] tensor; with an
    fp32 block scale tensor (a checkpoint that was not re-quantized) this is the ordinary block-FP8 linear, the
    reference's fallback."""
    assert input_scale is None
    if weight_scale.dtype != torch.int32 or input.dtype != torch.bfloat16 or weight.shape[1] % 128 != 0:
        return triton_w8a8_block_fp8_linear(input, weight, block_size, weight_scale, input_scale, bias)
    if not is_dynamo_compiling():
        out = _native.try_block_linear_ue8m0(input, weight, block_size, weight_scale, bias)
        if out is not None:
            return out
    from .fp8_kernel import sglang_per_token_group_quant_fp8

    K = input.shape[-1]
    x2d = input.reshape(-1, K)
    if not x2d.is_contiguous():
        x2d = x2d.contiguous()
    one_call = (list(block_size) == [128, 128] and x2d.is_cuda and x2d.shape[0] > 0 and weight.dim() == 2
                and weight.is_contiguous() and weight.dtype == torch.float8_e4m3fn and weight.shape[1] == K
                and weight_scale.dim() == 2 and weight_scale.shape[0] == weight.shape[0]
                and weight_scale.shape[1] >= (K // 128 + 3) // 4)
    if one_call:  # the same quantizer and GEMM kernels on the same data behind one C-ABI call
        out = ops.block_fp8_linear_ue8m0(x2d, weight, weight_scale, None, input.dtype)
    else:
        q_input, x_scale = sglang_per_token_group_quant_fp8(
            x2d, block_size[1], column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True, enable_v2=True)
        out = w8a8_block_fp8_matmul_deepgemm(q_input, weight, x_scale, weight_scale, block_size, output_dtype=input.dtype)
    if bias is not None:
        out += bias
    return out.to(dtype=input.dtype).view(*input.shape[:-1], weight.shape[0])


def apply_fp8_linear(
    input: torch.Tensor,
    weight: torch.Tensor,
    weight_scale: torch.Tensor,
    input_scale: Optional[torch.Tensor] = None,
    input_scale_ub: Optional[torch.Tensor] = None,
    bias: Optional[torch.Tensor] = None,
    cutlass_fp8_supported: bool = True,
    use_per_token_if_dynamic: bool = False,
    pad_output: Optional[bool] = None,
    compressed_tensor_quant: bool = False,
) -> torch.Tensor:
    """Per-token x per-channel FP8 linear (fp8_utils.py:565-853, the `fp8_scaled_mm` branches :627-640 / :786-808):
    `weight` is [K, N] column-major (the checkpoint's [N, K] transposed, as the reference keeps it), `weight_scale` has
    N elements (or one, for a per-tensor weight scale, which is expanded).  Activations: dynamic per-token scales by
    default; a static per-tensor `input_scale` is repeated per token (:748-753); with `compressed_tensor_quant` the
    quantizer is `scaled_fp8_quant` (:598-603), whose per-tensor scale is repeated likewise for the GEMM.
    `input_scale_ub` is accepted and unused, as in the reference (:570 is its only mention there)."""
    if not compressed_tensor_quant and not is_dynamo_compiling():
        out = _native.try_token_linear(input, weight, weight_scale, input_scale, bias)
        if out is not None:
            return out
    K = input.shape[-1]
    N = weight.shape[1]
    x2d = input.reshape(-1, K)
    if not x2d.is_contiguous():
        x2d = x2d.contiguous()
    if compressed_tensor_quant:
        q, s = scaled_fp8_quant(x2d, input_scale, use_per_token_if_dynamic=use_per_token_if_dynamic)
        if s.numel() == 1:
            s = s.reshape(1, 1).expand(x2d.shape[0], 1).contiguous()
    elif input_scale is not None:
        assert input_scale.numel() == 1
        q, s = static_quant_fp8(x2d, input_scale, repeat_scale=True)
    else:
        q = None  # dynamic per-token scales: one call below where its preconditions hold
    ws = weight_scale.reshape(-1).to(torch.float32)
    if ws.numel() == 1:
        ws = ws.expand(N)
    ws = ws.contiguous()
    if q is None:
        one_call = (x2d.is_cuda and x2d.shape[0] > 0 and input.dtype in (torch.bfloat16, torch.float16) and weight.dim() == 2
                    and weight.dtype == torch.float8_e4m3fn and weight.stride(0) == 1 and weight.shape[0] == K and K % 16 == 0
                    and N % 8 == 0 and ws.numel() == N
                    and (bias is None or (bias.dtype == input.dtype and bias.is_contiguous() and bias.numel() == N)))
        if one_call:  # the same two kernels on the same data behind one C-ABI call
            return ops.fp8_per_token_linear(x2d, weight, ws, bias, input.dtype).view(*input.shape[:-1], N)
        q, s = sglang_per_token_quant_fp8(x2d)
    out = fp8_scaled_mm(q, weight, s, ws, out_dtype=input.dtype, bias=bias)
    return out.view(*input.shape[:-1], N)


# ---------------------------------------------------------------- weight side: 128 x 128 block (re)quantization at load time

def ceil_div(a: int, b: int) -> int:
    return (a + b - 1) // b


def per_block_cast_to_fp8(x: torch.Tensor):
    """fp8_utils.py:487-500: 128 x 128 blocks, power-of-two scales (ceil_to_ue8m0), amax floored at 1e-4."""
    assert x.dim() == 2
    return ops.block_cast_to_fp8(x)


def block_quant_dequant(x_q_block: torch.Tensor, x_s: torch.Tensor, block_size: List[int], dtype: torch.dtype) -> torch.Tensor:
    """fp8_utils.py:392-413 for 128 x 128 blocks; leading batch dimensions are walked one matrix at a time."""
    assert list(block_size) == [128, 128], "only 128 x 128 blocks are built"
    *batch, n, k = x_q_block.shape
    if not batch:
        return ops.block_dequant_fp8(x_q_block, x_s, dtype)
    q3, s3 = x_q_block.reshape(-1, n, k), x_s.reshape(-1, ceil_div(n, 128), ceil_div(k, 128))
    out = torch.stack([ops.block_dequant_fp8(q3[i], s3[i], dtype) for i in range(q3.shape[0])])
    return out.view(*batch, n, k)


def quant_weight_ue8m0(weight_dequant: torch.Tensor, weight_block_size: List[int]):
    """fp8_utils.py:452-478: bf16 weight [..., n, k] -> (e4m3fn weight, fp32 power-of-two scales [..., n/128, k/128])."""
    assert list(weight_block_size) == [128, 128]
    assert weight_dequant.dtype == torch.bfloat16, f"{weight_dequant.dtype=} {weight_dequant.shape=}"
    *batch_dims, n, k = weight_dequant.shape
    out_w_flat, out_s_flat = per_block_cast_to_fp8(weight_dequant.reshape(-1, k))
    out_w = out_w_flat.view((*batch_dims, n, k))
    out_s = out_s_flat.view((*batch_dims, ceil_div(n, 128), ceil_div(k, 128)))
    return out_w, out_s


def transform_scale_ue8m0(sf: torch.Tensor, mn: int) -> torch.Tensor:
    """fp8_utils.py:485-491 (`_transform_scale_ue8m0`): one scale row per weight row (index_select by row // 128), then
    the packed layout DeepGEMM's `get_mn_major_tma_aligned_packed_ue8m0_tensor` produces - exponent bytes, four per int32
    along k, words MN-major with the MN extent padded to a multiple of four - i.e. the layout
    create_per_token_group_quant_fp8_output_scale(scale_ue8m0=True) allocates for activations.  DeepGEMM itself is not
    part of the reference tree; the layout is the one its callers in the reference rely on."""
    *batch, _, kb = sf.shape
    rows = torch.arange(mn, device=sf.device) // 128
    per_row = sf.index_select(-2, rows)                                   # [..., mn, kb] fp32 powers of two
    expo = (per_row.contiguous().view(torch.int32) >> 23).to(torch.uint8)   # exponent byte
    kw = ceil_div(kb, 4)
    padded = torch.zeros((*batch, mn, kw * 4), dtype=torch.uint8, device=sf.device)
    padded[..., :kb] = expo
    words = padded.view(torch.int32)                                        # [..., mn, kw], little endian: byte j = group 4w + j
    aligned_mn = ceil_div(mn, 4) * 4
    out = torch.zeros((*batch, kw, aligned_mn), dtype=torch.int32, device=sf.device)
    out[..., :mn] = words.transpose(-1, -2)
    return out.transpose(-1, -2)[..., :mn, :]


def requant_weight_ue8m0(weight: torch.Tensor, weight_scale_inv: torch.Tensor, weight_block_size: List[int]):
    """fp8_utils.py:428-449 (`_requant_weight_ue8m0`): dequantize a block-FP8 weight to bf16, quantize it again with
    power-of-two block scales, return (weight, packed UE8M0 scales)."""
    assert list(weight_block_size) == [128, 128]
    weight_dequant = block_quant_dequant(weight, weight_scale_inv, weight_block_size, torch.bfloat16)
    out_w, out_s = quant_weight_ue8m0(weight_dequant=weight_dequant, weight_block_size=weight_block_size)
    return out_w, transform_scale_ue8m0(out_s, mn=out_w.shape[-2])
