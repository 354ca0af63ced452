"""Preparation and tile choice of the grouped FP8 GEMM at the edges of what they do: experts that end inside, at and behind a 32-row
chunk, several experts and none in one, more experts than one scan takes, K of a part of 32 blocks, one expert with all rows;
64 and 128 token by 128 and 256 channel tiles, alone and behind the 256-row tiles."""
import pytest
import torch

from gemm_cases import GROUPED_FORMS
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


@pytest.mark.parametrize("E,rows,N,K", [form[:4] for form in GROUPED_FORMS])
def test_every_tiling(gpu, oracle, E, rows, N, K):
    print(f"case {E} {rows} {N} {K}", flush=True)
    g = torch.Generator().manual_seed(E + rows)
    weight = torch.rand(E, generator=g) + 0.1
    weight[E // 2] += E / 4
    if E > 2:
        weight[1] = 0
    sizes = torch.bincount(torch.multinomial(weight, rows, replacement=True, generator=g), minlength=E).tolist()
    a, w, sa, sw, offsets, T = _problem(sizes, N, K, rows + N)
    out = _call(gpu, a, w, sa, sw, sizes, offsets, torch.bfloat16)
    _verify(oracle, out, a, w, sa, sw, sizes, offsets, f"{E} {rows}")


# routing that is not dense and in order, on the one-launch tile and where tables are prepared: (sizes, offsets, stacked rows, N, K, what runs)
SHARED = [([40, 40, 24], [0, 20, 80], 104, 256, 256, "grouped_wavesplit"), ([40, 40, 24], [0, 20, 80], 104, 6152, 256, "grouped_dma3"),
          # out of order, one inside another, one outside every 32-row chunk of the others, a gap inside a chunk
          ([30, 7, 50, 3], [60, 64, 5, 200], 237, 264, 384, "grouped_wavesplit"), ([30, 7, 50, 3], [60, 64, 5, 200], 237, 5128, 384, "grouped_dma3")]
# more experts than a scan takes at a time: rows shared inside the second 256 experts, and with one of the first
MANY = [1] * 300
MANY_OFFSETS = [e + (e > 100) * 3 for e in range(300)]
MANY[280], MANY[281], MANY_OFFSETS[290] = 5, 3, 10
SHARED += [(MANY, MANY_OFFSETS, 310, 24, 128, "grouped_wavesplit"), (MANY, MANY_OFFSETS, 310, 1032, 128, "grouped_dma3")]


@pytest.mark.parametrize("sizes,offsets,T,N,K,kernel", SHARED, ids=lambda v: str(v) if isinstance(v, (int, str)) else str(len(v)))
def test_experts_that_share_rows(gpu, oracle, sizes, offsets, T, N, K, kernel):
    """Overlapping offsets: every expert still multiplies the rows it names with its own weight; rows named by several hold results of
    theirs, and rows named by none stay as they were.  Prepared scales have a column for each row of an expert, which two that share rows
    may share too: wrong results there are what such routing gets, and nowhere else."""
    from sglang_amd import _lib

    print(f"case {T} {N} {K} {_lib.grouped_gemm_plan(len(sizes), T, N, K)}", flush=True)
    assert _lib.grouped_gemm_plan(len(sizes), T, N, K)["kernel"] == kernel
    a, w, sa, sw, _, _ = _problem([T] + [0] * (len(sizes) - 1), N, K, 5)
    out = _call(gpu, a, w, sa, sw, sizes, offsets, torch.bfloat16).float().cpu()
    right, owners = torch.zeros(T, N, dtype=torch.bool), torch.zeros(T, dtype=torch.int32)
    column = lambda e, r0: (r0 + 3) // 4 * 4 + 4 * e
    taken = torch.zeros(2 * T + 4 * len(sizes), dtype=torch.int32)
    for e, (m, r0) in enumerate(zip(sizes, offsets)):
        taken[column(e, r0):column(e, r0) + m] += 1
    own_scales = torch.ones(T, dtype=torch.bool)
    for e, (m, r0) in enumerate(zip(sizes, offsets)):
        rows = slice(r0, r0 + m)
        own_scales[rows] &= taken[column(e, r0):column(e, r0) + m] == 1
        ref, mag = oracle.fp8_blockwise_mm(a[rows], w[e], sa[rows], sw[e], torch.float32, want_abs=True)
        right[rows] |= (out[rows] - ref).abs() <= 1e-2 * ref.abs() + 1e-4 * mag
        owners[rows] += 1
    assert bool((owners > 1).any()) and bool((owners == 0).any())
    if kernel == "grouped_wavesplit":
        own_scales[:] = True
    assert 2 * int((own_scales & (owners > 0)).sum()) > int((owners > 0).sum())
    assert bool(right[own_scales & (owners > 0)].all()) and bool((out[owners == 0] == 7.0).all())


@pytest.mark.parametrize("N,kernel", [(256, "grouped_wavesplit"), (5128, "grouped_dma3")])
def test_gaps_and_sizes_beyond_the_matrix(gpu, oracle, N, kernel):
    """Unused rows between experts, some of them in the same 32 as used ones, and a last expert that claims more rows than there are."""
    from sglang_amd import _lib

    sizes = [5, 100, 0, 33, 64]
    a, w, sa, sw, offsets, T = _problem(sizes, N, 512, 9, gap=7)
    assert _lib.grouped_gemm_plan(5, T, N, 512)["kernel"] == kernel
    _verify(oracle, _call(gpu, a, w, sa, sw, sizes, offsets, torch.float16), a, w, sa, sw, sizes, offsets, "gaps")
    claimed, there = sizes[:4] + [1 << 20], sizes[:4] + [T - offsets[4]]
    _verify(oracle, _call(gpu, a, w, sa, sw, claimed, offsets, torch.float16), a, w, sa, sw, there, offsets, "claimed")
    # offsets outside the matrix: nothing of those experts is written
    beyond = offsets[:3] + [-4, T + 9]
    out = _call(gpu, a, w, sa, sw, sizes[:3] + [0, 64], beyond, torch.float16)
    _verify(oracle, out, a, w, sa, sw, sizes[:3] + [0, 0], offsets, "beyond")


@pytest.mark.parametrize("sizes,N,K,kernel", [([70, 9, 140], 512, 640, "grouped_wavesplit"), ([70, 9, 140], 4104, 640, "grouped_dma3"),
                                              ([200, 1, 77, 300, 0, 129], 384, 768, "grouped_wavesplit"),
                                              ([200, 1, 77, 300, 0, 129], 2056, 768, "grouped_dma3")])
def test_entry_points_and_scale_layouts_agree(gpu, sizes, N, K, kernel):
    """Both entry points, and token scales row-major and column-major: the same bits."""
    from sglang_amd import _lib
    from sglang_amd.sgl_kernel import es_fp8_blockwise_scaled_grouped_mm

    a, w, sa, sw, offsets, T = _problem(sizes, N, K, 21)
    E = len(sizes)
    assert _lib.grouped_gemm_plan(E, T, N, K)["kernel"] == kernel
    want = _call(gpu, a, w, sa, sw, sizes, offsets, torch.bfloat16)
    assert torch.equal(want, _call(gpu, a, w, sa.to(gpu).t().contiguous().t(), sw, sizes, offsets, torch.bfloat16))
    out = torch.full((T, N), 7.0, dtype=torch.bfloat16, device=gpu)
    i64 = lambda v: torch.full((E,), v, dtype=torch.int64, device=gpu)
    es_fp8_blockwise_scaled_grouped_mm(
        out, a.to(gpu), w.to(gpu).transpose(1, 2), sa.to(gpu), sw.to(gpu).transpose(1, 2), i64(K), i64(K), i64(N),
        torch.tensor([[m, N, K] for m in sizes], dtype=torch.int32, device=gpu),
        torch.tensor(offsets, dtype=torch.int32, device=gpu), torch.empty(16 << 20, dtype=torch.uint8, device=gpu))
    assert torch.equal(want, out)
