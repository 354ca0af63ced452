"""Every variant that the four GEMMs run (block scales, packed exponents, one scale per token and channel, INT8), at a shape of
tests/gemm_cases.py that reaches it, and the mid-M tiles with every remainder of the K blocks over their LDS stages.  Small-integer operands
and power-of-two scales: every product, block sum and partial sum is exact in fp32 in any order, so a stale stage, a block
multiplied twice or skipped, a wrong scale or a wrong row shows as a wrong number.  The reference is the product in float64."""
import pytest
import torch

from gemm_cases import MID_TILE_SWEEPS, VARIANT_SHAPES, plan_for, variant_of

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


def check_exact(gpu, kind, M, N, K):
    from sglang_amd import ops

    g = torch.Generator(device=gpu).manual_seed(M + 3 * N + 5 * K)
    draw = lambda low, high, *shape: torch.randint(low, high, shape, generator=g, device=gpu)
    a, w = draw(-2, 3, M, K), draw(-2, 3, N, K)
    kb, nb = -(-K // 128), -(-N // 128)
    if kind in ("fp8", "fp8_ue8m0"):
        ea, eb = draw(125, 130, M, kb), draw(125, 130, nb, kb)
        ta, tb = torch.exp2(ea.double() - 127), torch.exp2(eb.double() - 127)
        wide = lambda s: s.repeat_interleave(128, dim=1)[:, :K]
        want = (a * wide(ta)) @ (w * wide(tb.repeat_interleave(128, dim=0)[:N])).t()
        a8, w8 = a.float().to(FP8), w.float().to(FP8)
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
            out = ops.fp8_scaled_mm(a.float().to(FP8), w.float().to(FP8).t(), sa, sb, torch.bfloat16, bias)
        else:
            a8, w8 = a.to(torch.int8), w.to(torch.int8)
            assert torch.equal(ops.int8_mm_raw_accumulators(a8, w8.t()).double(), product), (kind, M, N, K)
            out = ops.int8_scaled_mm(a8, w8.t(), sa, sb, torch.bfloat16, bias)
    assert torch.equal(out, want.float().to(torch.bfloat16)), (kind, M, N, K)


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
