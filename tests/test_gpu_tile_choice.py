"""Every tile of the modelled choice (wave-split tiles, and mid-M tiles the constants table does not name) at ragged sizes: token
and channel counts that are no multiples of it, K of fewer blocks than a workgroup has waves and of remainders of its turns, and,
where only the epilogue scales, K in multiples of 16.  Small-integer operands with power-of-two scales are exact in fp32 in any
order, so every arithmetic must give the exact result."""
import pytest
import torch

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn

# (M, N, K), tile of the block-scaled FP8 GEMM, tile of the INT8 GEMM (None: the plan's own)
CASES = [((17, 136, 384), (16, 16), (16, 16)), ((33, 1544, 384), (16, 32), (16, 32)), ((33, 4104, 384), (16, 64), (16, 64)),
         ((17, 2056, 384), (32, 16), (32, 16)), ((17, 4104, 384), (32, 32), (32, 32)), ((17, 8200, 640), (32, 64), None),
         ((33, 3080, 384), (48, 16), (48, 16)), ((33, 6152, 640), (48, 32), (48, 32)), ((49, 4104, 1152), (64, 32), (64, 32)),
         ((33, 8200, 2304), (64, 64), None), ((33, 8200, 3200), None, (64, 64)), ((1, 136, 2304), (16, 16), (16, 16)),
         ((16, 9224, 1152), (16, 64), (16, 64)), ((15, 4168, 8320), (16, 32), (16, 32)), ((257, 8200, 384), (64, 192), None),
         ((193, 12296, 384), (64, 128), None), ((385, 8200, 640), (64, 256), None), ((129, 12296, 1152), None, (96, 128)),
         ((193, 8200, 384), None, (64, 128)), ((1000, 2056, 384), None, (64, 192)), ((385, 12296, 384), (96, 256), (96, 256)),
         ((1000, 4104, 384), (96, 192), (96, 192)), ((500, 8200, 384), (192, 128), (192, 128)), ((500, 8200, 640), None, (128, 192)),
         ((700, 6152, 384), (160, 128), (160, 128)), ((700, 8200, 384), None, (160, 192)), ((65, 8200, 7168), (96, 128), None)]
RAGGED_K = [(1, 136, 400), (17, 520, 4112), (33, 264, 16), (64, 1032, 912), (90, 2056, 5920), (5, 264, 784), (400, 328, 976)]


def _pow2(shape, g, low=-3, high=4):
    return torch.exp2(torch.randint(low, high, shape, generator=g).float())


def _words(e, rows):
    """exponent bytes [rows, groups] -> int32 words [rows, ceil(groups / 4)] with stride 1 along the rows (pitch in whole fours)"""
    groups = e.shape[1]
    buf = torch.zeros((groups + 3) // 4, (rows + 3) // 4 * 4, dtype=torch.int32)
    for k in range(groups):
        buf[k // 4, :rows] |= torch.from_numpy((e[:, k].numpy().astype("uint32") << (8 * (k % 4))).view("int32"))
    return buf


@pytest.mark.parametrize("shape,fp8_tile,int8_tile", CASES + [(s, None, None) for s in RAGGED_K])
def test_every_tile_exact(gpu, shape, fp8_tile, int8_tile):
    from sglang_amd import _lib, ops
    from sglang_amd.sgl_kernel import fp8_scaled_mm, int8_scaled_mm

    M, N, K = shape
    for kind, tile in (("fp8", fp8_tile), ("int8", int8_tile)):
        plan = _lib.gemm_plan(kind, M, N, K)
        print(f"case {kind} {shape} {plan}", flush=True)
        if tile is not None:
            assert (plan["bm"], plan["bn"]) == tile
    g = torch.Generator().manual_seed(M + N + K)
    a, w = torch.randint(-2, 3, (M, K), generator=g), torch.randint(-2, 3, (N, K), generator=g)
    a8, w8 = a.float().to(FP8).to(gpu), w.float().to(FP8).to(gpu)
    product = a.double() @ w.double().T
    sa, sb = _pow2((M,), g), _pow2((N,), g)
    bias = torch.randint(-16, 17, (N,), generator=g).float().to(torch.bfloat16)
    want = product * sa.double()[:, None] * sb.double()[None, :] + bias.double()[None, :]
    out = fp8_scaled_mm(a8, w8.t(), sa.to(gpu), sb.to(gpu), torch.bfloat16, bias.to(gpu))
    assert torch.equal(out.cpu(), want.to(torch.float32).to(torch.bfloat16))
    out = int8_scaled_mm(a.to(torch.int8).to(gpu), w.to(torch.int8).to(gpu).t(), sa.to(gpu), sb.to(gpu), torch.bfloat16, bias.to(gpu))
    assert torch.equal(out.cpu(), want.to(torch.float32).to(torch.bfloat16))
    acc = ops.int8_mm_raw_accumulators(a.to(torch.int8).to(gpu), w.to(torch.int8).to(gpu).t())
    assert torch.equal(acc.cpu().double(), product)
    if K % 128:
        return
    kb, nb = K // 128, -(-N // 128)
    ea, eb = torch.randint(125, 130, (M, kb), generator=g), torch.randint(125, 130, (nb, kb), generator=g)
    ta, tb = torch.exp2(ea.double() - 127), torch.exp2(eb.double() - 127)
    want = torch.zeros(M, N, dtype=torch.float64)
    for k in range(kb):
        part = a[:, 128 * k:128 * k + 128].double() @ w[:, 128 * k:128 * k + 128].double().T
        want += part * ta[:, k:k + 1] * tb[:, k].repeat_interleave(128)[None, :N]
    want = want.to(torch.float32).to(torch.bfloat16)
    for scales in (ta.float().to(gpu), ta.float().t().contiguous().to(gpu).t()):  # K-major and M-major token scales
        out = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
        ops.block_fp8_matmul(a8, w8, scales, tb.float().to(gpu), out)
        assert torch.equal(out.cpu(), want)
    out = ops.fp8_blockwise_mm_ue8m0(a8, w8, _words(ea, M).to(gpu).t()[:M], _words(eb.repeat_interleave(128, 0)[:N], N).to(gpu).t()[:N], torch.bfloat16)
    assert torch.equal(out.cpu(), want)
