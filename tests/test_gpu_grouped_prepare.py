"""Preparation and tile choice of the grouped FP8 GEMM at the edges of what they do: experts that end inside, at and behind a 32-row
chunk, several experts and none in one, more experts than one scan takes, K of a part of 32 blocks, one expert with all rows;
64 and 128 token by 128 and 256 channel tiles, alone and behind the 256-row tiles."""
import pytest
import torch

from test_gpu_fp8_grouped_gemm import _call, _problem, _verify

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,sizes,N,K", [
    ("chunk_edges", [31, 1, 32, 33, 0, 0, 63, 1, 1, 64, 5], 384, 4480),
    ("all_rows_in_one", [0, 0, 0, 777, 0], 256, 640),
    ("two_scans", [1, 0, 2] * 110, 136, 128),
    ("one_row_each", [1] * 70, 512, 4224),
    ("wide", [40] * 16, 2056, 256),
    ("tall_and_wide", [160] * 8, 3000, 128),
    ("big_tiles", [700, 300, 129, 128, 1025], 2048, 4224),
    # the same edges with more channels, where tables are prepared
    ("chunk_edges_prepared", [31, 1, 32, 33, 0, 0, 63, 1, 1, 64, 5], 2056, 4480),
    ("two_scans_prepared", [1, 0, 2] * 110, 1032, 128),
    ("one_row_each_prepared", [1] * 70, 1040, 4224),
    # more experts than threads: runs of two a thread
    ("runs_of_experts", [0, 0, 0, 1, 2, 0] * 7 + [0] * 555 + [17, 3, 2], 24, 256),
])
@pytest.mark.parametrize("m_major", [False, True])
def test_grouped(gpu, oracle, name, sizes, N, K, m_major):
    print(f"case {name} {m_major}", flush=True)
    a, w, sa, sw, offsets, T = _problem(sizes, N, K, len(sizes) + N)
    scales = sa.to(gpu).t().contiguous().t() if m_major else sa
    out = _call(gpu, a, w, scales, sw, sizes, offsets, torch.bfloat16)
    _verify(oracle, out, a, w, sa, sw, sizes, offsets, name)


# experts (uneven: some without a row, one with many), stacked rows, N, K -> what has to run
FORMS = [(40, 1240, 2056, 128, "grouped_dma3", "64x256"), (2, 3254, 328, 384, "grouped_dma3", "64x128"),
         (16, 16, 64, 384, "grouped_wavesplit", "16x16"), (8, 209, 416, 128, "grouped_wavesplit", "16x32"), (40, 29, 392, 1152, "grouped_wavesplit", "16x64"),
         (5, 56, 1240, 128, "grouped_wavesplit", "32x32"), (40, 492, 272, 128, "grouped_wavesplit", "32x64"), (40, 1798, 136, 128, "grouped_wavesplit", "64x64"),
         (24, 1574, 128, 128, "grouped_wavesplit", "16x64"), (16, 1613, 224, 128, "grouped_wavesplit", "64x64"), (3, 545, 1544, 1152, "grouped_dma3", "64x128"),
         (40, 29, 2056, 128, "grouped_dma3", "64x128"),  # (more workgroups than CUs: two share one)
         (24, 1233, 2056, 384, "grouped_dma3", "128x256"), (16, 2075, 2056, 384, "grouped_dma3", "128x256"),
         (1, 1695, 2056, 640, "grouped_dma3", "128x128"), (24, 3078, 768, 2048, "grouped_dma3", "128x128"),
         (2, 5548, 2056, 384, "grouped_pingpong+grouped_dma3", "128x256")]


@pytest.mark.parametrize("E,rows,N,K,kernel,tile", FORMS)
def test_every_tiling(gpu, oracle, E, rows, N, K, kernel, tile):
    from sglang_amd import _lib

    plan = _lib.grouped_gemm_plan(E, rows, N, K)
    print(f"case {E} {rows} {N} {K} {plan}", flush=True)
    assert (plan["kernel"], plan["small_tile"]) == (kernel, tile)
    g = torch.Generator().manual_seed(E + rows)
    weight = torch.rand(E, generator=g) + 0.1
    weight[E // 2] += E / 4
    if E > 2:
        weight[1] = 0
    sizes = torch.bincount(torch.multinomial(weight, rows, replacement=True, generator=g), minlength=E).tolist()
    a, w, sa, sw, offsets, T = _problem(sizes, N, K, rows + N)
    out = _call(gpu, a, w, sa, sw, sizes, offsets, torch.bfloat16)
    _verify(oracle, out, a, w, sa, sw, sizes, offsets, f"{E} {rows}")


def test_experts_that_share_rows(gpu, oracle):
    """Overlapping offsets: every expert still multiplies the rows it names with its own weight; rows named twice hold the result of
    one of them."""
    sizes = [40, 40, 24]
    a, w, sa, sw, _, T = _problem(sizes, 256, 256, 5)
    out = _call(gpu, a, w, sa, sw, sizes, [0, 20, 80], torch.bfloat16).float().cpu()
    for e, (m, r0) in enumerate(zip(sizes, (0, 20, 80))):
        ref, mag = oracle.fp8_blockwise_mm(a[r0:r0 + m], w[e], sa[r0:r0 + m], sw[e], torch.float32, want_abs=True)
        alone = [r for r in range(r0, r0 + m) if not 20 <= r < 40]
        index = torch.tensor(alone) - r0
        assert bool(((out[alone] - ref[index]).abs() <= 1e-2 * ref[index].abs() + 1e-4 * mag[index]).all())
