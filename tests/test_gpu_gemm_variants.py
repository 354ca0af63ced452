"""Every variant that the four GEMMs run (block scales, packed exponents, one scale per token and channel, INT8), at a shape of
tests/gemm_cases.py that reaches it (held by the CPU tests), and the mid-M tiles with every remainder of the K blocks over their LDS stages.  Small-integer operands
and power-of-two scales: every product, block sum and partial sum is exact in fp32 in any order, so a stale stage, a block
multiplied twice or skipped, a wrong scale or a wrong row shows as a wrong number.  The reference is the product in float64."""
import pytest
import torch

from gemm_cases import MID_TILE_SWEEPS, TAKEN_OVER_SHAPES, VARIANT_SHAPES, plan_for, variant_of

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn


def _words(e):
    """exponent bytes [rows, groups] -> int32 words [rows, ceil(groups / 4)] with stride 1 along the rows (pitch in whole fours)"""
    rows, groups = e.shape
    full = torch.zeros(rows, (groups + 3) // 4 * 4, dtype=torch.uint8, device=e.device)
    full[:, :groups] = e.to(torch.uint8)
    buf = torch.zeros((groups + 3) // 4, (rows + 3) // 4 * 4, dtype=torch.int32, device=e.device)
    buf[:, :rows] = full.view(torch.int32).t()
    return buf.t()[:rows]


def check_exact(gpu, kind, M, N, K, pitch=None, behind=1, token_pitch=None):
    """`pitch`: elements between the weight's rows, with the bytes `behind` after each (127 is a NaN as FP8); `token_pitch`: between the tokens'."""
    from sglang_amd import ops

    g = torch.Generator(device=gpu).manual_seed(M + 3 * N + 5 * K)
    draw = lambda low, high, *shape: torch.randint(low, high, shape, generator=g, device=gpu)
    a, w = draw(-2, 3, M, K), draw(-2, 3, N, K)
    kb, nb = -(-K // 128), -(-N // 128)
    pad = lambda t: torch.nn.functional.pad(t, (0, pitch - K), value=behind)[:, :K] if pitch else t

    def apart(t):
        if token_pitch is None:
            return t
        rows = torch.empty((M - 1) * token_pitch + K, dtype=torch.uint8, device=gpu).as_strided((M, K), (token_pitch, 1))
        return rows.copy_(t.view(torch.uint8)).view(t.dtype)

    if kind in ("fp8", "fp8_ue8m0"):
        ea, eb = draw(125, 130, M, kb), draw(125, 130, nb, kb)
        ta, tb = torch.exp2(ea.double() - 127), torch.exp2(eb.double() - 127)
        wide = lambda s: s.repeat_interleave(128, dim=1)[:, :K]
        want = (a * wide(ta)) @ (w * wide(tb.repeat_interleave(128, dim=0)[:N])).t()
        a8, w8 = a.float().to(FP8), pad(w.float().to(FP8).view(torch.uint8)).view(FP8)
        if kind == "fp8":
            out = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
            ops.block_fp8_matmul(a8, w8, ta.float(), tb.float(), out)
        else:
            out = ops.fp8_blockwise_mm_ue8m0(a8, w8, _words(ea), _words(eb.repeat_interleave(128, dim=0)[:N]), torch.bfloat16)
    else:
        sa, sb = torch.exp2(draw(-3, 4, M).float()), torch.exp2(draw(-3, 4, N).float())
        bias = draw(-16, 17, N).to(torch.bfloat16)
        product = a.double() @ w.double().t()
        want = product * sa.double()[:, None] * sb.double() + bias.double()
        if kind == "fp8_scaled":
            out = ops.fp8_scaled_mm(apart(a.float().to(FP8)), pad(w.float().to(FP8).view(torch.uint8)).view(FP8).t(), sa, sb, torch.bfloat16, bias)
        else:
            a8, w8 = apart(a.to(torch.int8)), pad(w.to(torch.int8))
            assert torch.equal(ops.int8_mm_raw_accumulators(a8, w8.t()).double(), product), (kind, M, N, K)
            out = ops.int8_scaled_mm(a8, w8.t(), sa, sb, torch.bfloat16, bias)
    assert torch.equal(out, want.float().to(torch.bfloat16)), (kind, M, N, K)


@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
@pytest.mark.parametrize("M,N,K", TAKEN_OVER_SHAPES)
def test_taken_over_exact(gpu, kind, M, N, K):
    print(f"case {kind} {(M, N, K)} {plan_for(kind, M, N, K)['kernel']}", flush=True)
    check_exact(gpu, kind, M, N, K)


@pytest.mark.parametrize("kind,variant", [(kind, v) for kind, shapes in VARIANT_SHAPES.items() for v in shapes],
                         ids=lambda x: x if isinstance(x, str) else "-".join(map(str, x)))
def test_variant_exact(gpu, kind, variant):
    M, N, K = VARIANT_SHAPES[kind][variant]
    print(f"case {kind} {(M, N, K)} {variant}", flush=True)
    assert variant_of(plan_for(kind, M, N, K), K) == variant
    check_exact(gpu, kind, M, N, K)


@pytest.mark.parametrize("kind,tile", [(kind, t) for kind, tiles in MID_TILE_SWEEPS.items() for t in tiles], ids=str)
def test_mid_tile_every_remainder(gpu, kind, tile):
    bm, bn, stages = tile
    M, N = MID_TILE_SWEEPS[kind][tile]
    for kb in range(1, 20):
        p = plan_for(kind, M, N, 128 * kb)
        if (p["kernel"], p["bm"], p["bn"], p["stages"], p["splits"]) == ("dma3", bm, bn, stages, 1):
            print(f"case {kind} {tile} {(M, N, 128 * kb)}", flush=True)
            check_exact(gpu, kind, M, N, 128 * kb)
            if kind == "fp8":  # (the same plan)
                assert plan_for("fp8_ue8m0", M, N, 128 * kb)["bm"] == bm
                check_exact(gpu, "fp8_ue8m0", M, N, 128 * kb)


# weight rows a multiple of 4096 bytes apart: every channel tile starts its K loop at another block (whole K and split, one and several
# token tiles, more channel tiles than K blocks and fewer, a ragged last tile)
@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
@pytest.mark.parametrize("M,N,K", [(40, 20480, 4096), (100, 15688, 4096), (100, 4096, 16384), (300, 8192, 8192), (23, 2184, 32768)])
def test_rotated_k(gpu, kind, M, N, K):
    assert N * K >= 64e6 and plan_for(kind, M, N, K)["kernel"] == "dma3"
    check_exact(gpu, kind, M, N, K)


# weight rows further apart than K bytes: 4096 bytes apart (K loops that start at different blocks, with streamed loads or without, decode
# sizes), and K = 4096 where they are not; the weight-in-registers kernel and the two-phase kernels
@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
@pytest.mark.parametrize("M,N,K,pitch", [(40, 20488, 3968, 4096), (300, 16392, 3968, 4096), (100, 28680, 3968, 4096), (8, 28688, 3968, 4096), (8, 28688, 4096, 4224),
                                         (100, 15688, 4096, 4224), (900, 16392, 512, 640), (1, 1040, 2176, 4096), (2100, 8200, 1024, 1152)])
def test_weight_rows_of_any_pitch(gpu, kind, M, N, K, pitch):
    print(f"case {kind} {(M, N, K)} pitch {pitch}", flush=True)
    check_exact(gpu, kind, M, N, K, pitch)


# tokens whose rows span more than 4 GiB stay on the kernel of 64-bit offsets, in tiles of 256 tokens with K split and whole
@pytest.mark.parametrize("kind", ["fp8_scaled", "int8"])
@pytest.mark.parametrize("M,N,K", [(1052, 6688, 928), (1052, 6688, 128), (70, 520, 1040)])
def test_token_rows_over_four_gigabytes(gpu, kind, M, N, K):
    check_exact(gpu, kind, M, N, K, token_pitch=(1 << 32) // M // 16 * 16 + 32)


# weights of 100 million bytes and more are loaded as a stream where one token tile reads them: every height of the mid-M tile, K split and
# whole, the 16-token tile, ragged last channel tiles
@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
@pytest.mark.parametrize("M,N,K", [(13, 7176, 14336), (64, 7176, 18432), (33, 9224, 11264), (40, 36872, 2816), (90, 24584, 4224), (150, 24584, 4224),
                                   (185, 28680, 3840)])
def test_streamed_weights(gpu, kind, M, N, K):
    p = plan_for(kind, M, N, K)
    assert N * K >= 1e8 and p["kernel"] in ("dma3", "wavesplit_tile") and M <= p["bm"]
    check_exact(gpu, kind, M, N, K)


# the same below the kernels that quantize the tokens themselves: their results are those of a quantizer launch and the GEMM
@pytest.mark.parametrize("M,N,K", [(2, 7184, 14336), (16, 24576, 7168), (7, 36880, 7168)])
def test_streamed_weights_of_fused_linears(gpu, M, N, K):
    from sglang_amd import _lib, ops
    from sglang_amd.fp8_kernel import per_token_group_quant_fp8, w8a8_block_fp8_matmul

    assert _lib.linear_plan("block", M, N, K)["quantizer"] == "fused" and N * K >= 1e8
    g = torch.Generator(device=gpu).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
    w = torch.randint(-8, 9, (N, K), generator=g, device=gpu, dtype=torch.int8).half().to(FP8)
    s = torch.rand((N + 127) // 128, K // 128, generator=g, device=gpu) + 0.5
    q, qs = per_token_group_quant_fp8(x, 128, column_major_scales=True)
    two = w8a8_block_fp8_matmul(q, w, qs, s, [128, 128], torch.bfloat16)
    assert torch.equal(ops.block_fp8_linear(x, w, s, None, torch.bfloat16).view(torch.int16), two.view(torch.int16))


def test_block_linear_on_padded_rows(gpu):
    """Rows 4096 bytes apart with K below that, and the other way round: what dense rows give, where the sums have one order, and the
    same to the rounding of the result where the K loops start at other blocks."""
    from fp8_tolerance import check_fp8_gemm
    from sglang_amd import ops
    from sglang_amd.fp8_kernel import per_token_group_quant_fp8

    for M, N, K, pitch in ((4, 28672, 3968, 4096), (16, 28672, 3968, 4096), (4, 28672, 4096, 4224), (1, 1024, 2176, 4096)):
        g = torch.Generator(device=gpu).manual_seed(M + K)
        x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
        w = torch.randint(-8, 9, (N, pitch), generator=g, device=gpu, dtype=torch.int8).half().to(FP8)[:, :K]
        s = torch.rand(N // 128, K // 128, generator=g, device=gpu) + 0.5
        out = ops.block_fp8_linear(x, w, s, None, torch.bfloat16)
        q, qs = per_token_group_quant_fp8(x, 128, column_major_scales=True)
        a = q.double() * qs.double().repeat_interleave(128, 1)
        b = w[:1024].double() * s[:8].double().repeat_interleave(128, 0).repeat_interleave(128, 1)
        check_fp8_gemm(out[:, :1024], (a @ b.t()).float().cpu(), (a.abs() @ b.abs().t()).float().cpu(), f"{(M, N, K, pitch)}")


# the block linear's own choice on such weights, also where the GEMM alone takes another kernel: the wave-split tile quantizing and behind a
# launch, producer waves, the mid-M tile where the rows lie 4096 bytes apart; the first and the last channels
@pytest.mark.parametrize("M,N,K", [(2, 16400, 9088), (1, 14352, 12672), (9, 14352, 8320), (16, 18448, 13312), (3, 40960, 3584), (5, 27904, 8192)])
def test_block_linear_on_streamed_weights(gpu, M, N, K):
    from fp8_tolerance import check_fp8_gemm
    from sglang_amd import _lib, ops
    from sglang_amd.fp8_kernel import per_token_group_quant_fp8

    print(f"case {(M, N, K)} {_lib.block_linear_plan(M, N, K)}", flush=True)
    assert _lib.block_linear_plan(M, N, K)["kernel"] in ("wavesplit_tile", "dma3")
    g = torch.Generator(device=gpu).manual_seed(M)
    x = torch.randn(M, K, generator=g, device=gpu).bfloat16()
    w = torch.randint(-8, 9, (N, K), generator=g, device=gpu, dtype=torch.int8).half().to(FP8)
    s = torch.rand((N + 127) // 128, K // 128, generator=g, device=gpu) + 0.5
    out = ops.block_fp8_linear(x, w, s, None, torch.bfloat16)
    q, qs = per_token_group_quant_fp8(x, 128, column_major_scales=True)  # (the linear's arithmetic: x / s)
    a = q.double() * qs.double().repeat_interleave(128, 1)
    for cols in (slice(0, 256), slice((N - 200) // 128 * 128, N)):
        rows = s[cols.start // 128:(cols.stop + 127) // 128].double().repeat_interleave(128, 0)[:cols.stop - cols.start]
        b = w[cols].double() * rows.repeat_interleave(128, 1)
        check_fp8_gemm(out[:, cols], (a @ b.t()).float().cpu(), (a.abs() @ b.abs().t()).float().cpu(), f"{(M, N, K)}")


# results on both sides of the size up to which they are written through the L2: the weight-in-registers and the two-phase kernels
@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
@pytest.mark.parametrize("N,K", [(32768, 256), (24584, 896), (8200, 1024)])
@pytest.mark.parametrize("more", [0, 1])
def test_results_written_through(gpu, kind, N, K, more):
    check_exact(gpu, kind, 64000000 // N + more, N, K)


# the same out of the mid-M, the 128-token and (K = 768) the weight-in-registers kernel, and with the kernel named where packed exponents go
# straight to the two-phase one
@pytest.mark.parametrize("kind,N,K,kernel", [("fp8", 13592, 128, "dma3"), ("fp8_ue8m0", 13592, 128, "dma3"), ("fp8_scaled", 65584, 128, "dma3"),
                                             ("int8", 65584, 768, "resident"),
                                             ("int8", 65584, 896, "pingpong128"), ("fp8_ue8m0", 24584, 1024, "pingpong")])
@pytest.mark.parametrize("more", [0, 1])
def test_results_written_through_by_kernel(gpu, kind, N, K, kernel, more):
    M = 64000000 // N + more
    assert plan_for(kind, M, N, K)["kernel"] == kernel
    check_exact(gpu, kind, M, N, K)


# weight in registers: more steps of tokens than the LDS has stages, a last range with fewer, channels that end inside a slice, and fewer
# tokens than a step
@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
@pytest.mark.parametrize("kb", [2, 3, 4, 5])
def test_resident_many_steps(gpu, kind, kb):
    for M, N in ((1237, 30008), (2049, 16392), (3000, 7176)):
        print(f"case {kind} {(M, N, 128 * kb)}", flush=True)
        assert plan_for(kind, M, N, 128 * kb)["kernel"] == "resident"
        check_exact(gpu, kind, M, N, 128 * kb)


@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
def test_resident_six_blocks(gpu, kind):
    """The longest K whose weight the registers hold: the sizes above, with and without results that are written through."""
    for M, N in ((1237, 30008), (2049, 16392), (2600, 24584), (3000, 7176)):
        print(f"case {kind} {(M, N, 768)}", flush=True)
        assert plan_for(kind, M, N, 768)["kernel"] == "resident"
        check_exact(gpu, kind, M, N, 768)


def test_resident_hands_over_outputs_it_cannot_store(gpu):
    """16-byte stores of 16-bit results: a base or a row pitch that does not allow them, and fp32 results, take another kernel."""
    import ctypes

    from sglang_amd import _lib

    M, N, K = 600, 16384, 512
    assert plan_for("fp8", M, N, K)["kernel"] == "resident"
    g = torch.Generator(device=gpu).manual_seed(1)
    a, w = (torch.randint(-2, 3, s, generator=g, device=gpu).float().to(FP8) for s in ((M, K), (N, K)))
    sa, sb = torch.ones(K // 128, M, device=gpu), torch.ones(N // 128, K // 128, device=gpu)
    want = a.double() @ w.double().t()
    ws = torch.empty(_lib.lib().mi355_fp8_blockwise_mm_workspace_bytes(M, N, K), dtype=torch.uint8, device=gpu)
    for code, dtype, pitch, shift in ((2, torch.bfloat16, N, 0), (2, torch.bfloat16, N, 4), (2, torch.bfloat16, N + 4, 0), (1, torch.float16, N + 8, 0), (0, torch.float32, N, 0)):
        out = torch.zeros(M * pitch + 64, dtype=dtype, device=gpu)
        ptr = lambda t: ctypes.c_void_p(t.data_ptr())
        rc = _lib.lib().mi355_fp8_blockwise_mm(ptr(a), ptr(w), ptr(sa), ptr(sb), ctypes.c_void_p(out.data_ptr() + shift * out.element_size()), code, M, N, K, K, K,
                                               1, M, K // 128, 1, pitch, ptr(ws), ws.numel(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, (dtype, pitch, shift, _lib.lib().mi355_last_error())
        rows = out[shift:shift + M * pitch].view(M, pitch)
        assert torch.equal(rows[:, :N].double(), want.to(dtype).double()), (dtype, pitch, shift)
        assert not out[:shift].any() and not out[shift + M * pitch:].any() and not rows[:, N:].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_resident_bias_and_rows(gpu, dtype):
    """The four linears with a bias: the rows that a smaller call, on another kernel with the same order of sums, computes."""
    from sglang_amd import _lib, fp8_utils, w8a8_int8
    from sglang_amd.workloads import make_activation, make_fp8_weight, make_int8_weight

    M, N, K = 900, 24576, 512
    x = make_activation(M, K, dtype=dtype).to(gpu)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(2)).to(dtype).to(gpu)
    w, s = (t.to(gpu) for t in make_fp8_weight(N, K))
    w2, words = fp8_utils.requant_weight_ue8m0(w, s, [128, 128])
    wi, si = (t.to(gpu) for t in make_int8_weight(N, K))
    scale = torch.rand(N, 1, generator=torch.Generator().manual_seed(3)).to(gpu) * 0.01 + 1e-3
    linear = fp8_utils.dispatch_w8a8_block_fp8_linear()
    calls = {"block": lambda x: linear(x, w, [128, 128], s, None, bias), "token_fp8": lambda x: fp8_utils.apply_fp8_linear(x, w.t(), scale, None, bias=bias, use_per_token_if_dynamic=True),
             "int8": lambda x: w8a8_int8.apply_w8a8_int8_linear(x, wi.t(), si, bias)}
    if dtype == torch.bfloat16:
        calls["ue8m0"] = lambda x: fp8_utils.deepgemm_w8a8_block_fp8_linear_with_fallback(x, w2, [128, 128], words, None, bias)
    for kind, call in calls.items():
        few = 200
        assert _lib.linear_plan(kind, M, N, K)["kernel"] == "resident" and _lib.linear_plan(kind, few, N, K)["kernel"] == "dma3"
        assert _lib.linear_plan(kind, few, N, K)["splits"] == 1
        assert torch.equal(call(x)[:few].view(torch.int16), call(x[:few].contiguous()).view(torch.int16)), kind


@pytest.mark.parametrize("kind", ["block", "ue8m0", "token_fp8", "int8"])
@pytest.mark.parametrize("kb", [2, 3, 4, 5, 6])
def test_resident_kinds_of_output(gpu, kind, kb):
    """A kernel for each output type, with and without a bias, written through or not (beyond 128 MB): channels that end inside a slice and tokens
    inside a half step, against the first and last rows by a smaller call, on another kernel with the same order of sums."""
    from sglang_amd import _lib, fp8_utils, w8a8_int8
    from sglang_amd.workloads import make_activation, make_fp8_weight, make_int8_weight

    N, K, few = 24584, 128 * kb, 40
    w, s = (t.to(gpu) for t in make_fp8_weight(N, K))
    w2, words = fp8_utils.requant_weight_ue8m0(w, s, [128, 128])
    wi, si = (t.to(gpu) for t in make_int8_weight(N, K))
    scale = torch.rand(N, 1, generator=torch.Generator().manual_seed(3)).to(gpu) * 0.01 + 1e-3
    linear = fp8_utils.dispatch_w8a8_block_fp8_linear()
    call = {"block": lambda x, b: linear(x, w, [128, 128], s, None, b), "ue8m0": lambda x, b: fp8_utils.deepgemm_w8a8_block_fp8_linear_with_fallback(x, w2, [128, 128], words, None, b),
            "token_fp8": lambda x, b: fp8_utils.apply_fp8_linear(x, w.t(), scale, None, bias=b, use_per_token_if_dynamic=True),
            "int8": lambda x, b: w8a8_int8.apply_w8a8_int8_linear(x, wi.t(), si, b)}[kind]
    assert _lib.linear_plan(kind, few, N, K)["kernel"] == "dma3" and _lib.linear_plan(kind, few, N, K)["splits"] == 1
    for M in (901, 2701):
        assert _lib.linear_plan(kind, M, N, K)["kernel"] == "resident" and (M * N * 2 <= 128000000) == (M == 901)
        for dtype in (torch.bfloat16,) if kind == "ue8m0" else (torch.bfloat16, torch.float16):
            x = make_activation(M, K, dtype=dtype).to(gpu)
            for bias in (None, torch.randn(N, generator=torch.Generator().manual_seed(2)).to(dtype).to(gpu)):
                out = call(x, bias)
                for rows in (slice(0, few), slice(M - few, M)):
                    assert torch.equal(out[rows].view(torch.int16), call(x[rows].contiguous(), bias).view(torch.int16)), (M, dtype, bias is not None, rows)


# wave-split tile, many more tokens than channels: the workgroups of an XCD take the channel tiles of the same tokens
@pytest.mark.parametrize("kind", ["fp8", "fp8_ue8m0", "fp8_scaled", "int8"])
@pytest.mark.parametrize("M,N,K", [(1003, 200, 1024), (2050, 136, 896), (1403, 312, 896)])
def test_more_tokens_than_channels(gpu, kind, M, N, K):
    check_exact(gpu, kind, M, N, K)


def test_more_tokens_than_channels_linears(gpu):
    from sglang_amd import fp8_utils, w8a8_int8
    from sglang_amd.workloads import make_activation, make_fp8_weight, make_int8_weight

    M, N, K = 517, 200, 512
    x = make_activation(M, K).to(gpu)
    w, s = (t.to(gpu) for t in make_fp8_weight(N, K))
    wi, si = (t.to(gpu) for t in make_int8_weight(N, K))
    linear = fp8_utils.dispatch_w8a8_block_fp8_linear()
    for call in (lambda x: linear(x, w, [128, 128], s, None, None), lambda x: w8a8_int8.apply_w8a8_int8_linear(x, wi.t(), si, None),
                 lambda x: fp8_utils.apply_fp8_linear(x, w.t(), torch.ones(N, 1, device=gpu), None, use_per_token_if_dynamic=True)):
        out = call(x)
        for first in range(0, M, 40):
            assert torch.equal(out[first:first + 40].view(torch.int16), call(x[first:first + 40].contiguous()).view(torch.int16)), first

