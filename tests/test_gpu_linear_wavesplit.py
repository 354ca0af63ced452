"""One-call linears whose wave-split kernels quantize the tokens themselves: at the steps of the pieces a thread quantizes
(2, 4, 10), four and eight waves, one and two channel tiles, K blocks that do not fill the waves' turns, and just past the
limit, where a quantizer launch stands in front of the GEMM again; and every other thing the four linears do (gemm_cases)."""
import pytest
import torch

from fp8_tolerance import check_fp8_gemm
from gemm_cases import LINEAR_SHAPES, QUANT_TILE_KERNELS, QUANT_TILE_SHAPES
from sglang_amd.workloads import make_activation, make_fp8_weight, make_int8_weight

pytestmark = pytest.mark.gpu

# pieces of 8 values per thread: M K / (8 * 64 * waves)
SHAPES = [(1, 4096, 1152), (8, 144, 2048), (16, 4096, 1152), (2, 576, 4096), (3, 1040, 2176), (4, 512, 4096), (5, 512, 4096),
          (10, 6144, 4096), (11, 512, 4096), (1, 512, 8320), (1, 272, 20480), (2, 40960, 4096), (5, 576, 7168)]


@pytest.mark.parametrize("M,N,K", SHAPES + [s for s in LINEAR_SHAPES if s not in SHAPES])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_quantizer_of_the_wavesplit_kernel(gpu, oracle, M, N, K, dtype):
    from sglang_amd import _lib, ops
    from sglang_amd.fp8_kernel import per_token_group_quant_fp8, sglang_per_token_group_quant_fp8, sglang_per_token_quant_fp8, w8a8_block_fp8_matmul
    from sglang_amd.fp8_utils import _one_call_takes_the_same_gemm, requant_weight_ue8m0
    from sglang_amd.int8_kernel import per_token_quant_int8

    print(f"case M={M} N={N} K={K} {[_lib.linear_plan(k, M, N, K) for k in ('block', 'ue8m0', 'token_fp8', 'int8')]}", flush=True)
    bits = lambda t: t.view(torch.int16)
    x = make_activation(M, K, seed=M + N, dtype=dtype)
    x[0, :128] = 0
    if M > 2:
        x[M - 1] = 0  # a token of zeros
    xg = x.to(gpu)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(N)).to(dtype).to(gpu)
    w_q, w_s = make_fp8_weight(N, K, seed=K)
    wg, sg = w_q.to(gpu), w_s.to(gpu)
    for by_reciprocal in (False, True):
        out = ops.block_fp8_linear(xg, wg, sg, None, dtype, by_reciprocal=by_reciprocal)
        q, s = per_token_group_quant_fp8(xg, 128, column_major_scales=not by_reciprocal)
        two = w8a8_block_fp8_matmul(q, wg, s, sg, [128, 128], dtype)
        if _one_call_takes_the_same_gemm(M, N, K):
            assert torch.equal(bits(out), bits(two))
        if N <= 1040:
            xq, xs = oracle.group_quant(x, 128, mode="rcp" if by_reciprocal else "div")
            ref, mag = oracle.fp8_blockwise_mm(xq, w_q, xs, w_s, torch.float32, want_abs=True)
            check_fp8_gemm(out, ref, mag, "block")
    w2, words = requant_weight_ue8m0(wg, sg, [128, 128])
    q, s = sglang_per_token_group_quant_fp8(xg, 128, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True)
    assert torch.equal(bits(ops.block_fp8_linear_ue8m0(xg, w2, words, bias, dtype)), bits(ops.fp8_blockwise_mm_ue8m0(q, w2, s, words, dtype, bias)))
    scale = torch.rand(N, generator=torch.Generator().manual_seed(K)).to(gpu) * 0.01 + 1e-3
    q, s = sglang_per_token_quant_fp8(xg)
    assert torch.equal(bits(ops.fp8_per_token_linear(xg, wg.t(), scale, bias, dtype)), bits(ops.fp8_scaled_mm(q, wg.t(), s, scale, dtype, bias)))
    i_q, i_s = make_int8_weight(N, K, seed=K)
    q, s = per_token_quant_int8(xg)
    iw, isc = i_q.to(gpu).t(), i_s.to(gpu)
    assert torch.equal(bits(ops.int8_linear(xg, iw, isc, bias, dtype)), bits(ops.int8_scaled_mm(q, iw, s, isc, dtype, bias)))


def test_reciprocal_on_every_significand(gpu):
    """RN(1 / s) and RN(s / 448) of the quantizers inside the GEMMs, for every float of the exponents that a scale (or, for the second, a
    group's maximum) can have: 1e-10 / 448 and up to the largest bfloat16."""
    import ctypes

    from sglang_amd import _lib

    counts = torch.zeros(2, dtype=torch.int64, device=gpu)
    for e in range(-43, 120):
        _lib.check(_lib.lib().mi355_probe_reciprocal(e, ctypes.c_void_p(counts.data_ptr()), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert counts.tolist() == [0, 0]
    assert _lib.lib().mi355_probe_reciprocal(121, ctypes.c_void_p(counts.data_ptr()), None) == 1


@pytest.mark.parametrize("tile,many", QUANT_TILE_SHAPES)
def test_fused_quantizer_above_decode_sizes(gpu, tile, many):
    """One launch against quantizer and GEMM entry point, which runs on a wave-split tile of its own size: the same codes, scales and sums,
    so the same results bit for bit, with rows that are all zero, infinite or partly NaN.  (Some of the four linears take the named tile; each
    tile by each linear is QUANT_TILE_KERNELS.)"""
    from sglang_amd import _lib, ops
    from sglang_amd.fp8_kernel import per_token_group_quant_fp8, sglang_per_token_group_quant_fp8, sglang_per_token_quant_fp8, w8a8_block_fp8_matmul
    from sglang_amd.fp8_utils import requant_weight_ue8m0
    from sglang_amd.int8_kernel import per_token_quant_int8

    M, N, K = QUANT_TILE_SHAPES[tile, many]
    plans = {k: _lib.linear_plan(k, M, N, K) for k in ("block", "ue8m0", "token_fp8", "int8")}
    print(f"case M={M} N={N} K={K} {plans}", flush=True)
    for dtype in (torch.bfloat16, torch.float16):
        bits = lambda t: torch.where(t.isnan(), torch.zeros_like(t), t).view(torch.int16)
        x = make_activation(M, K, seed=M + N, dtype=dtype)
        x[0], x[M - 1], x[M // 2, 5], x[1, 7] = 0, 0, float("inf"), float("nan")
        xg = x.to(gpu)
        bias = torch.randn(N, generator=torch.Generator().manual_seed(N)).to(dtype).to(gpu)
        w_q, w_s = make_fp8_weight(N, K, seed=K)
        wg, sg = w_q.to(gpu), w_s.to(gpu)
        for by_reciprocal in (False, True):
            q, s = per_token_group_quant_fp8(xg, 128, column_major_scales=not by_reciprocal)
            out, two = ops.block_fp8_linear(xg, wg, sg, None, dtype, by_reciprocal=by_reciprocal), w8a8_block_fp8_matmul(q, wg, s, sg, [128, 128], dtype)
            assert torch.equal(bits(out), bits(two)) and torch.equal(out.isnan(), two.isnan())
        w2, words = requant_weight_ue8m0(wg, sg, [128, 128])
        q, s = sglang_per_token_group_quant_fp8(xg, 128, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True, enable_v2=True)
        out, two = ops.block_fp8_linear_ue8m0(xg, w2, words, bias, dtype), ops.fp8_blockwise_mm_ue8m0(q, w2, s, words, dtype, bias)
        assert torch.equal(bits(out), bits(two)) and torch.equal(out.isnan(), two.isnan())
        scale = torch.rand(N, generator=torch.Generator().manual_seed(K)).to(gpu) * 0.01 + 1e-3
        q, s = sglang_per_token_quant_fp8(xg)
        out, two = ops.fp8_per_token_linear(xg, wg.t(), scale, bias, dtype), ops.fp8_scaled_mm(q, wg.t(), s, scale, dtype, bias)
        assert torch.equal(bits(out), bits(two)) and torch.equal(out.isnan(), two.isnan())
        xg[M // 2, 5] = xg[1, 7] = 1  # (a row with an infinity has no INT8 codes)
        i_q, i_s = make_int8_weight(N, K, seed=K)
        q, s = per_token_quant_int8(xg)
        iw, isc = i_q.to(gpu).t(), i_s.to(gpu)
        assert torch.equal(bits(ops.int8_linear(xg, iw, isc, bias, dtype)), bits(ops.int8_scaled_mm(q, iw, s, isc, dtype, bias)))


@pytest.mark.parametrize("kind,kernel,shape", [(kind, kernel, shape) for kinds, *kernel, shape in QUANT_TILE_KERNELS for kind in kinds.split()],
                         ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_kernel_that_quantizes_in_its_tile(gpu, kind, kernel, shape, dtype):
    """Small integers whose groups (rows) have a maximum of 448 (127) times a power of two: scales are powers of two, codes the values, and sums
    exact in any order.  Padded weight rows hold NaN bytes (127) behind K; a row's last value is its maximum.  The kernel that a shape
    runs is held by the CPU tests."""
    from sglang_amd import ops
    from test_gpu_gemm_variants import _words

    M, N, K = shape
    print(f"case {kind} {kernel} {shape} {dtype}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M + 3 * N + 5 * K)
    draw = lambda low, high, *s: torch.randint(low, high, s, generator=g, device=gpu)
    most, kb, nb = 127 if kind == "int8" else 448, -(-K // 128), -(-N // 128)
    v = draw(-3, 4, M, K).double()
    if kind in ("block", "ue8m0"):
        v.view(M, kb, 128)[:, :, 127] = most * (1 - 2 * draw(0, 2, M, kb))
        v = (v.view(M, kb, 128) * torch.exp2(draw(-2, 3, M, kb).double())[:, :, None]).reshape(M, K)
    else:
        v[:, K - 1] = most * (1 - 2 * draw(0, 2, M))
        v = v * torch.exp2(draw(-2, 3, M).double())[:, None]
    x = v.to(dtype)
    assert torch.equal(x.double(), v)
    pitch = (K + 127) // 128 * 128
    codes = torch.full((N, pitch), 127, dtype=torch.uint8, device=gpu)  # (NaN as FP8)
    wv = draw(-2, 3, N, K)
    codes[:, :K] = (wv.to(torch.int8) if kind == "int8" else wv.half().to(torch.float8_e4m3fn)).view(torch.uint8)
    w = codes.view(torch.int8 if kind == "int8" else torch.float8_e4m3fn)[:, :K]
    if kernel[4] == "cached" and K % 128:  # dense rows: the next row's bytes lie behind K
        w = w.contiguous()
    if kind in ("block", "ue8m0"):
        eb = draw(125, 130, nb, kb)
        full = torch.exp2(eb.double() - 127).repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)[:, :K]
        want = v @ (wv * full).t()
        out = ops.block_fp8_linear(x, w, torch.exp2(eb.float() - 127), None, dtype) if kind == "block" else \
            ops.block_fp8_linear_ue8m0(x, w, _words(eb.repeat_interleave(128, dim=0)[:N]), None, dtype)
    else:
        sb = torch.exp2(draw(-3, 4, N).float())
        want = (v @ wv.double().t()) * sb.double()
        out = (ops.int8_linear if kind == "int8" else ops.fp8_per_token_linear)(x, w.t(), sb, None, dtype)
    assert torch.equal(out, want.float().to(dtype))


# every kernel that quantizes tokens itself: (kinds, kernel, channel tile or waves, shape)
FUSED_KERNELS = [(("block", "block_rcp", "ue8m0", "token_fp8", "int8"), "wavesplit_tile", 0, (16, 2176, 2176)),
                 (("block", "block_rcp", "ue8m0", "token_fp8", "int8"), "wavesplit_tile", 0, (16, 1024, 512)),
                 (("block", "block_rcp", "ue8m0", "token_fp8", "int8"), "decode_wavesplit", 4, (4, 7168, 2048)),
                 (("block", "block_rcp", "ue8m0", "token_fp8", "int8"), "decode_wavesplit", 8, (1, 16512, 3840)),
                 (("block", "block_rcp"), "decode", 1, (16, 16896, 512)), (("block", "block_rcp"), "decode", 1, (13, 20864, 1536)),
                 (("block", "block_rcp"), "dma3", 128, (16, 24576, 1536)), (("block", "block_rcp"), "dma3", 192, (13, 45056, 1280)),
                 (("block", "block_rcp"), "dma3", 256, (13, 53248, 1152))]


@pytest.mark.parametrize("kind,kernel,detail,M,N,K", [(kind, k, d, *s) for kinds, k, d, s in FUSED_KERNELS for kind in kinds])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_quantizer_on_every_16_bit_value(gpu, kind, dtype, kernel, detail, M, N, K):
    """Every bit pattern (infinities and NaN among them) through a one-hot weight: a channel's result is one code times its scales,
    so the quantizer inside the GEMM has to write the codes and scales of the quantizer kernels."""
    from sglang_amd import _lib, ops
    from sglang_amd.fp8_kernel import per_token_group_quant_fp8, sglang_per_token_group_quant_fp8, sglang_per_token_quant_fp8, w8a8_block_fp8_matmul
    from sglang_amd.fp8_utils import requant_weight_ue8m0
    from sglang_amd.int8_kernel import per_token_quant_int8

    plan = _lib.linear_plan(kind.split("_rcp")[0], M, N, K)
    assert plan["quantizer"] == "fused" and plan["kernel"] == kernel and detail in (0, plan["bn" if kernel == "dma3" else "groups_per_wg"]), plan
    calls = -(-65536 // (M * K))
    patterns = torch.randperm(65536, generator=torch.Generator().manual_seed(3))
    patterns = torch.cat([patterns, torch.zeros(calls * M * K - 65536, dtype=torch.int64)]).to(torch.int32).to(torch.int16).view(calls, M, K)
    # a second pair of inputs, all finite and sorted: groups of one magnitude, where the rounding of every quotient shows
    finite = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(dtype)
    finite = finite[torch.isfinite(finite)].float().sort().values.to(dtype)
    finite = torch.cat([finite, torch.zeros(calls * M * K - finite.numel(), dtype=dtype)]).view(calls, M, K)
    w = torch.zeros(N, K, device=gpu, dtype=torch.float16)
    w[torch.arange(N), torch.arange(N) % K] = 1
    one, ones = torch.ones(N, device=gpu), torch.ones(N // 128, K // 128, device=gpu)
    for x in [*patterns.view(dtype), *finite]:
        if kind == "ue8m0":  # (the two quantizers of this kind clamp a NaN to different ends)
            x = torch.nan_to_num(x, nan=0.0, posinf=float("inf"), neginf=float("-inf"))
        xg = x.contiguous().to(gpu)
        if kind == "int8":
            wi = w.to(torch.int8).t()
            q, s = per_token_quant_int8(xg)
            out, two = ops.int8_linear(xg, wi, one, None, dtype), ops.int8_scaled_mm(q, wi, s, one, dtype, None)
        elif kind == "token_fp8":
            wf = w.to(torch.float8_e4m3fn).t()
            q, s = sglang_per_token_quant_fp8(xg)
            out, two = ops.fp8_per_token_linear(xg, wf, one, None, dtype), ops.fp8_scaled_mm(q, wf, s, one, dtype, None)
        elif kind == "ue8m0":
            w2, words = requant_weight_ue8m0(w.to(torch.float8_e4m3fn), ones, [128, 128])
            q, s = sglang_per_token_group_quant_fp8(xg, 128, column_major_scales=True, scale_tma_aligned=True, scale_ue8m0=True, enable_v2=True)
            out, two = ops.block_fp8_linear_ue8m0(xg, w2, words, None, dtype), ops.fp8_blockwise_mm_ue8m0(q, w2, s, words, dtype, None)
        else:
            wf, rcp = w.to(torch.float8_e4m3fn), kind == "block_rcp"
            q, s = per_token_group_quant_fp8(xg, 128, column_major_scales=not rcp)
            out, two = ops.block_fp8_linear(xg, wf, ones, None, dtype, by_reciprocal=rcp), w8a8_block_fp8_matmul(q, wf, s, ones, [128, 128], dtype)
        same = (out.view(torch.int16) == two.view(torch.int16)) | (out.isnan() & two.isnan())
        assert bool(same.all()), (~same).sum().item()
