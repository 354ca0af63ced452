"""K in parts of 128-value blocks on the mid-M tile (INT8, and FP8 with one scale per token and channel): every tile and pipeline depth,
last blocks of 16 to 112 values, fewer K blocks than stages, ragged last tiles.  Small-integer operands with power-of-two scales are exact
in fp32 in any order, so the result has to be exact; a channel of NaN has to stay in its own column, whatever its row's neighbours read."""
import pytest
import torch

pytestmark = pytest.mark.gpu
FP8 = torch.float8_e4m3fn

# (M, N, K) and the tile it runs on
CASES = [((17, 17208, 272), (64, 128)), ((17, 36192, 272), (64, 128)), ((17, 36192, 400), (64, 192)), ((33, 17208, 656), (64, 128)), ((20, 16392, 6160), (64, 128)), ((17, 45656, 304), (64, 192)),
         ((396, 8888, 1456), (64, 256)), ((71, 18736, 400), (96, 128)), ((70, 33408, 272), (96, 192)), ((272, 16456, 288), (96, 256)), ((97, 24888, 928), (128, 128)),
         ((207, 17048, 288), (128, 192)), ((215, 25152, 272), (128, 256)), ((133, 24744, 352), (160, 128)), ((136, 35040, 272), (160, 192)),
         ((331, 12432, 368), (192, 128)), ((667, 10824, 272), (256, 128)), ((3, 15000, 6704), None)]


@pytest.mark.parametrize("shape,tile", CASES)
def test_parts_of_blocks_exact(gpu, shape, tile):
    from sglang_amd import _lib
    from sglang_amd.sgl_kernel import fp8_scaled_mm, int8_scaled_mm

    M, N, K = shape
    for kind in ("fp8_scaled", "int8"):
        plan = _lib.gemm_plan(kind, M, N, K)
        print(f"case {kind} {shape} {plan}", flush=True)
        if tile is not None:
            assert plan["kernel"] == "dma3" and (plan["bm"], plan["bn"]) == tile
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
