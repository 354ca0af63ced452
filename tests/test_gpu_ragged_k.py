"""K in parts of 128-value blocks on the mid-M tile (INT8, and FP8 with one scale per token and channel): every tile and pipeline depth,
last blocks of 16 to 112 values, fewer K blocks than stages, ragged last tiles.  Small-integer operands with power-of-two scales are exact
in fp32 in any order, so the result has to be exact; a channel of NaN has to stay in its own column, whatever its row's neighbours read.
The tile that each shape runs is held by the CPU tests."""
import pytest
import torch

from gemm_cases import RAGGED_TILE_SHAPES, STREAMED_RAGGED_SHAPES

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn

SHAPES = [shape for shape, _ in RAGGED_TILE_SHAPES] + [(3, 15000, 6704), (65, 25352, 912), (1052, 6688, 928)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_parts_of_blocks_exact(gpu, shape):
    from sglang_amd import _lib
    from sglang_amd.sgl_kernel import fp8_scaled_mm, int8_scaled_mm

    M, N, K = shape
    print(f"case {shape} {_lib.gemm_plan('int8', M, N, K)}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    a, w = torch.randint(-2, 3, (M, K), generator=g, device=gpu), torch.randint(-2, 3, (N, K), generator=g, device=gpu)
    sa = torch.exp2(torch.randint(-3, 4, (M,), generator=g, device=gpu).float())
    sb = torch.exp2(torch.randint(-3, 4, (N,), generator=g, device=gpu).float())
    product = a.float() @ w.float().T  # |sums| below 2^24: exact
    want = (product * sa[:, None] * sb[None, :]).to(torch.bfloat16)
    out = int8_scaled_mm(a.to(torch.int8), w.to(torch.int8).t(), sa, sb, torch.bfloat16)
    assert torch.equal(out, want)
    w8 = w.float().to(FP8)
    out = fp8_scaled_mm(a.float().to(FP8), w8.t(), sa, sb, torch.bfloat16)
    assert torch.equal(out, want)
    w8[5] = torch.full((K,), float("nan"), device=gpu).to(FP8)
    out = fp8_scaled_mm(a.float().to(FP8), w8.t(), sa, sb, torch.bfloat16)
    assert out[:, 5].isnan().all()
    keep = torch.arange(N, device=gpu) != 5
    assert torch.equal(out[:, keep], want[:, keep])


@pytest.mark.parametrize("kind", ["fp8_scaled", "int8"])
@pytest.mark.parametrize("shape", [shape for shape, _ in STREAMED_RAGGED_SHAPES], ids=str)
def test_streamed_parts_of_blocks_exact(gpu, kind, shape):
    from test_gpu_gemm_variants import check_exact

    print(f"case {kind} {shape}", flush=True)
    check_exact(gpu, kind, *shape, pitch=(shape[2] + 127) // 128 * 128, behind=127)


# last blocks of 16 to 112 values, one block, rows that share a DPP row of sixteen pieces with no other, several token tiles, the most values a
# tile quantizes (40960); every kernel that does it: QUANT_TILE_KERNELS in gemm_cases.py
QUANTIZED = [(1, 136, 16), (3, 264, 112), (16, 576, 144), (5, 1032, 4112), (6, 2056, 6768), (16, 16400, 304), (45, 264, 272), (66, 264, 1200), (33, 4104, 1008), (2, 520, 20464), (16, 520, 1520),
             (700, 320, 368), (100, 4000, 272)]


@pytest.mark.parametrize("M,N,K", QUANTIZED)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_quantizer_inside_parts_of_blocks(gpu, M, N, K, dtype):
    """One launch against quantizer and GEMM entry point: the same codes, scales and sums, so the same bits, with zeros, infinities and NaN
    in some rows and at their ends; a static scale of zero too, whose codes are all at the limit."""
    from sglang_amd import _lib, ops
    from sglang_amd.fp8_kernel import sglang_per_token_quant_fp8, static_quant_fp8
    from sglang_amd.fp8_utils import apply_fp8_linear
    from sglang_amd.int8_kernel import per_token_quant_int8
    from sglang_amd.workloads import make_activation, make_fp8_weight, make_int8_weight

    for kind in ("token_fp8", "int8"):
        plan = _lib.linear_plan(kind, M, N, K)
        print(f"case {kind} {(M, N, K)} {plan}", flush=True)
        assert plan["quantizer"] == "fused"
    bits = lambda t: torch.where(t.isnan(), torch.zeros_like(t), t).view(torch.int16)
    whole = (K + 127) // 128 * 128
    x = make_activation(M, whole, seed=M + N, dtype=dtype)[:, :K].contiguous()
    if M > 2:
        x[0], x[M // 2, 5], x[1, K - 1] = 0, float("inf"), float("nan")
    x[M - 1, K - 1] = 300  # the row's maximum where it ends
    xg = x.to(gpu)
    w = make_fp8_weight(N, whole, seed=K)[0][:, :K].contiguous().to(gpu)
    scale = torch.rand(N, generator=torch.Generator().manual_seed(K)).to(gpu) * 0.01 + 1e-3
    bias = torch.randn(N, generator=torch.Generator().manual_seed(N)).to(dtype).to(gpu)
    q, s = sglang_per_token_quant_fp8(xg)
    out, two = ops.fp8_per_token_linear(xg, w.t(), scale, bias, dtype), ops.fp8_scaled_mm(q, w.t(), s, scale, dtype, bias)
    assert torch.equal(bits(out), bits(two)) and torch.equal(out.isnan(), two.isnan())
    for given in (0.5, 0.0):
        s = torch.tensor([given], device=gpu)
        q, rows = static_quant_fp8(xg, s, repeat_scale=True)
        out, two = apply_fp8_linear(xg, w.t(), scale, s, bias=bias), ops.fp8_scaled_mm(q, w.t(), rows, scale, dtype, bias)
        assert torch.equal(bits(out), bits(two)) and torch.equal(out.isnan(), two.isnan())
    if M > 2:
        xg[M // 2, 5] = xg[1, K - 1] = 1  # (a row with an infinity has no INT8 codes)
    q, s = per_token_quant_int8(xg)
    w8, ws = make_int8_weight(N, whole, seed=K)
    w8, ws = w8[:, :K].contiguous().to(gpu).t(), ws.to(gpu)
    assert torch.equal(bits(ops.int8_linear(xg, w8, ws, bias, dtype)), bits(ops.int8_scaled_mm(q, w8, s, ws, dtype, bias)))
