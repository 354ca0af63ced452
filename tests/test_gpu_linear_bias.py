"""The bias of the block-FP8 linears in the GEMM's epilogue: the bits of `output += bias`, whichever kernel runs (wave-split and
streaming decode kernels with and without a quantizer, mid-M tiles, split K, two-phase, generic), and a separate addition where
the bias is tracked by autograd or has another type."""
import pytest
import torch

from sglang_amd.workloads import make_activation, make_fp8_weight

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(1, 576, 7168), (3, 7168, 2048), (8, 1024, 512), (8, 24576, 1536), (12, 2048, 7168), (40, 200, 384),
                                   (33, 1536, 4096), (64, 7168, 18432), (300, 8192, 1152), (257, 24576, 1536), (2048, 8192, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_bias_in_the_epilogue(gpu, M, N, K, dtype):
    from sglang_amd import _lib
    from sglang_amd.fp8_utils import (cutlass_w8a8_block_fp8_linear_with_fallback, deepgemm_w8a8_block_fp8_linear_with_fallback,
                                      requant_weight_ue8m0, triton_w8a8_block_fp8_linear)

    print(f"case M={M} N={N} K={K} {dtype} {_lib.block_linear_plan(M, N, K)}", flush=True)
    x = make_activation(M, K, seed=M + N, dtype=dtype).to(gpu)
    w_q, w_s = (t.to(gpu) for t in make_fp8_weight(N, K, seed=K))
    bias = torch.randn(N, generator=torch.Generator().manual_seed(N)).to(dtype).to(gpu)
    w2, words = requant_weight_ue8m0(w_q, w_s, [128, 128])
    for linear, w, s in ((cutlass_w8a8_block_fp8_linear_with_fallback, w_q, w_s), (triton_w8a8_block_fp8_linear, w_q, w_s),
                         (deepgemm_w8a8_block_fp8_linear_with_fallback, w2, words)):
        if linear is deepgemm_w8a8_block_fp8_linear_with_fallback and dtype != torch.bfloat16:
            continue
        want = linear(x, w, [128, 128], s)
        want += bias
        assert torch.equal(linear(x, w, [128, 128], s, bias=bias).view(torch.int16), want.view(torch.int16))
        tracked = bias.clone().requires_grad_(True)
        out = linear(x, w, [128, 128], s, bias=tracked)
        assert out.requires_grad and torch.equal(out.detach().view(torch.int16), want.view(torch.int16))
