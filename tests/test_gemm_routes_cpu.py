"""Which kernel variant the dispatcher picks is a host-side decision, so it is checked without a GPU: the shapes the
GPU parity tests run (tests/gemm_cases.py) must between them reach every compiled variant, and the full-size benchmark
configurations must only use variants that those tests (or the full-size tests themselves) exercise."""
import random
import time

import pytest

from gemm_cases import (CAPTURED_LINEARS, FP8_DECODE_CONFIG, FP8_PREFILL_CONFIG, FP8_REQUIRED_VARIANTS, FP8_ROUTE_SHAPES, GROUPED_FORMS, GROUPED_SHAPES,
                        INT8_CONFIG, INT8_REQUIRED_VARIANTS, INT8_ROUTE_SHAPES, LINEAR_SHAPES, MID_TILE_SWEEPS, QUANT_TILE_KERNELS, QUANT_TILE_SHAPES, RAGGED_TILE_SHAPES,
                        STREAMED_RAGGED_SHAPES, VARIANT_SHAPES, linear_variant_of, plan_for, quant_tile_kernel, variant_of)

LINEARS = ("block", "ue8m0", "token_fp8", "int8")


def _reached(kind, shapes):
    return {variant_of(plan_for(kind, *s), s[2]) for s in shapes}


@pytest.mark.parametrize("kind", VARIANT_SHAPES)
def test_variant_shapes_run_what_they_are_named_after(kind):
    for variant, shape in VARIANT_SHAPES[kind].items():
        assert variant_of(plan_for(kind, *shape), shape[2]) == variant, (kind, shape)


@pytest.mark.parametrize("kind", VARIANT_SHAPES)
@pytest.mark.parametrize("kb", [2, 3, 4, 5, 6])
def test_resident_plan_names_the_tokens_of_a_step(kind, kb):
    """64 tokens a step of the weight-in-registers kernel, 32 where the registers hold no more beside the weight: from five K blocks on,
    with packed exponents from four on (whatever the other kinds' plan for the same shape was before)."""
    M, N, K = VARIANT_SHAPES[kind]["resident", f"kb{kb}"]
    for other in VARIANT_SHAPES:
        plan_for(other, M, N, K)
    assert plan_for(kind, M, N, K)["bm"] == (64 if kb <= (3 if kind == "fp8_ue8m0" else 4) else 32)


def _random_shapes(count, seed):
    """Token counts, channels and K over the whole range, half of the channels and three quarters of K in whole 128s."""
    import random

    rng = random.Random(seed)
    while count > 0:
        M, N, K = int(2 ** rng.uniform(0, 12.3)), int(2 ** rng.uniform(3, 16.2)), int(2 ** rng.uniform(4, 14.2))
        N = (N + 127) // 128 * 128 if rng.random() < 0.5 else (N + 7) // 8 * 8
        r = rng.random()
        K = (K + 127) // 128 * 128 if r < 0.75 else (K + 15) // 16 * 16 if r < 0.95 else K
        if N * K > 4.2e8:
            continue
        count -= 1
        yield M, N, K


def test_random_shapes_run_only_listed_variants():
    """A variant that the dispatcher learns to run has to get a shape in gemm_cases, or this fails."""
    for M, N, K in _random_shapes(6000, seed=17):
        for kind, listed in VARIANT_SHAPES.items():
            if K % (1 if kind == "fp8" else 128 if kind == "fp8_ue8m0" else 16) == 0:
                v = variant_of(plan_for(kind, M, N, K), K)
                assert v in listed, f"{kind} {(M, N, K)} runs {v}"


def test_random_linears_run_only_listed_variants():
    from sglang_amd import _lib

    listed = {kind: {linear_variant_of(_lib.linear_plan(kind, *s), s[0]) for s in LINEAR_SHAPES} for kind in LINEARS}
    for M, N, K in _random_shapes(4000, seed=18):
        M, K = (M - 1) % 20 + 1, (K + 127) // 128 * 128
        for kind in LINEARS:
            v = linear_variant_of(_lib.linear_plan(kind, M, N, K), M)
            assert v in listed[kind], f"{kind} {(M, N, K)} runs {v}"


def test_grouped_shapes_run_the_named_tiles():
    from sglang_amd import _lib

    for name, sizes, N, K, tile in GROUPED_SHAPES:
        assert _lib.grouped_gemm_plan(len(sizes), sum(sizes), N, K)["small_tile"] == tile, name
    for E, rows, N, K, kernel, tile in GROUPED_FORMS:
        plan = _lib.grouped_gemm_plan(E, rows, N, K)
        assert (plan["kernel"], plan["small_tile"]) == (kernel, tile), (E, rows, N, K)


@pytest.mark.parametrize("kind", ["fp8_scaled", "int8"])
def test_parts_of_blocks_run_the_named_tiles(kind):
    for shape, tile in RAGGED_TILE_SHAPES:
        p = plan_for(kind, *shape)
        assert ("dma3", 1, *tile) == (p["kernel"], p["splits"], p["bm"], p["bn"], p["stages"]), (shape, p)
    for shape, kernel in STREAMED_RAGGED_SHAPES:
        p = plan_for(kind, *shape)
        assert kernel == (p["kernel"], p["bm"], p["bn"]) and p["splits"] == 1 and shape[0] <= p["bm"] and shape[1] * shape[2] >= 1e8, (shape, p)


@pytest.mark.parametrize("tile,many", QUANT_TILE_SHAPES)
def test_quantizing_tiles_above_decode_sizes(tile, many):
    from sglang_amd import _lib

    M, N, K = QUANT_TILE_SHAPES[tile, many]
    plans = [_lib.linear_plan(kind, M, N, K) for kind in LINEARS]
    assert any((p["quantizer"], p["bm"], p["bn"]) == ("fused", *tile) for p in plans), plans
    assert (min(M, tile[0]) * K > (16384 if tile[0] == 16 else 20480)) == many


def test_quantizing_tiles_are_named_and_listed():
    """QUANT_TILE_KERNELS: each shape runs the kernel it stands for, and random linears run no other."""
    from sglang_amd import _lib

    listed = {kind: set() for kind in LINEARS}
    for kinds, *kernel, shape in QUANT_TILE_KERNELS:
        for kind in kinds.split():
            assert quant_tile_kernel(_lib.linear_plan(kind, *shape), *shape) == tuple(kernel), (kind, shape)
            listed[kind].add(tuple(kernel))
    rng = random.Random(31)
    spread = lambda low, high: int(low * (high / low) ** rng.random())
    for _ in range(20000):
        M, N, K = (spread(1, 16) if rng.random() < 0.5 else spread(17, 1200)), 8 * spread(1, 30000), 16 * spread(1, 2600)
        K = (K + 127) // 128 * 128 if rng.random() < 0.5 else K
        for kind in LINEARS if K % 128 == 0 else LINEARS[2:]:
            if N * K < 8e8:
                kernel = quant_tile_kernel(_lib.linear_plan(kind, M, N, K), M, N, K)
                assert kernel is None or kernel in listed[kind], f"{kind} {(M, N, K)} runs {kernel}"


def test_mid_tile_sweeps_meet_every_remainder():
    """Each mid-M tile, unsplit, with every remainder of the K blocks over its LDS stages (what the sweeps of the GPU test run)."""
    for kind, tiles in MID_TILE_SWEEPS.items():
        for (bm, bn, stages), (M, N) in tiles.items():
            assert {kb % stages for kb in _sweep(kind, bm, bn, stages, M, N)} == set(range(stages)), (kind, bm, bn, M, N)


def _sweep(kind, bm, bn, stages, M, N):
    plans = {kb: plan_for(kind, M, N, 128 * kb) for kb in range(1, 20)}
    return [kb for kb, p in plans.items() if (p["kernel"], p["bm"], p["bn"], p["stages"], p["splits"]) == ("dma3", bm, bn, stages, 1)]


def test_benchmark_configurations_use_only_tested_variants():
    for kind, config, routes, required in (("fp8", FP8_DECODE_CONFIG + FP8_PREFILL_CONFIG, FP8_ROUTE_SHAPES, FP8_REQUIRED_VARIANTS),
                                           ("int8", INT8_CONFIG, INT8_ROUTE_SHAPES, INT8_REQUIRED_VARIANTS)):
        tested = _reached(kind, routes + list(VARIANT_SHAPES[kind].values()))
        for s in config:
            v = variant_of(plan_for(kind, *s), s[2])
            assert v in tested and v in required, f"{kind} {s} runs {v}, which no route shape covers"


def test_every_variant_is_one_the_library_can_name():
    # a variant added to the dispatcher must be added to the required sets, or this fails
    for kind, shapes, required in (("fp8", FP8_ROUTE_SHAPES + FP8_DECODE_CONFIG + FP8_PREFILL_CONFIG, FP8_REQUIRED_VARIANTS),
                                   ("int8", INT8_ROUTE_SHAPES + INT8_CONFIG, INT8_REQUIRED_VARIANTS)):
        extra = _reached(kind, shapes) - required
        assert not extra, f"{kind}: variants reached but not listed as required: {sorted(extra, key=str)}"


# Kernel, tile and split alternatives that a +-10 % change of one constant reaches on a benchmark shape, with the median time of
# each in microseconds on MI355X (GEMM alone; ten launches over rotated weights in a graph, all alternatives in turn, the
# alternative forced by a build of the dispatcher whose plan is overridden).  The first entry of each shape is the dispatcher's own choice.
# A boundary is acceptable when both sides of it cost about the same.
RECORDED_BOUNDARIES = {
    ("fp8", (1, 7168, 18432)): {("wavesplit_tile", 16, 32, 1): 24.4, ("decode_wavesplit", 16, 32, 1): 24.8},
    ("fp8", (8, 7168, 18432)): {("wavesplit_tile", 16, 32, 1): 25.6, ("decode_wavesplit", 16, 32, 1): 28.0},
    ("fp8", (128, 7168, 18432)): {("dma3", 128, 128, 4): 44.2, ("dma3", 64, 128, 2): 49.8, ("dma3", 128, 192, 6): 43.1},
    ("fp8", (4096, 576, 7168)): {("dma3", 64, 192, 1): 31.2, ("dma3", 96, 128, 1): 31.3},
    ("int8", (1, 28672, 4096)): {("decode_wavesplit", 16, 16, 1): 23.2, ("dma3", 64, 128, 1): 21.8},
    ("int8", (256, 28672, 4096)): {("pingpong128", 128, 256, 1): 44.9, ("dma3", 128, 256, 1): 43.7},
    ("int8", (256, 4096, 14336)): {("dma3", 128, 128, 4): 32.6, ("wavesplit_tile", 64, 64, 1): 34.2},
    ("int8", (4096, 6144, 4096)): {("pingpong", 256, 256, 1): 100.7, ("dma3", 256, 128, 1): 97.6, ("dma3", 128, 256, 1): 101.2},
}
# The slower side of a recorded boundary may cost at most this much more than the dispatcher's choice: the widest one is 12.7 %
# (128 tokens on 18432 -> 7168, where 128 x 128 tiles became 10 % faster than when the older constants were drawn).
BOUNDARY_COST = 1.13


def test_benchmark_shapes_hold_their_kernels_when_a_constant_moves():
    """Every measured constant of the dispatcher's time models (sglang_amd/csrc/route_constants.h and tile_choice.h) is changed by
    -10 % and +10 %, one at a time.  A benchmark shape may move to another kernel, tile or split only where both have been
    timed on the GPU and recorded above, and the recorded times must show that the move costs less than BOUNDARY_COST: then the
    constant's uncertainty (timings spread +-3 %) cannot cost more than that.  A new constant, or a changed one, that puts a
    benchmark shape on an unmeasured boundary fails here."""
    from sglang_amd import _lib

    names = list(_lib.route_constants())
    assert len(names) == _lib.lib().mi355_route_constant_count() and len(set(names)) == len(names)
    tile = lambda p: (p["kernel"], p["bm"], p["bn"], p["splits"])
    moved = set()
    for kind, config in (("fp8", FP8_DECODE_CONFIG + FP8_PREFILL_CONFIG), ("int8", INT8_CONFIG)):
        for shape in config:
            base = plan_for(kind, *shape)
            for i, name in enumerate(names):
                for factor in (0.9, 1.1):
                    p = _lib.gemm_plan_perturbed(kind, *shape, i, factor)
                    if tile(p) == tile(base):
                        continue
                    rec = RECORDED_BOUNDARIES.get((kind, shape))
                    assert rec is not None and tile(base) in rec and tile(p) in rec, \
                        f"{kind} {shape}: {name} x {factor} moves tile {tile(base)} -> {tile(p)}: time both and record them"
                    assert next(iter(rec)) == tile(base), f"{kind} {shape}: the recorded choice {next(iter(rec))} is not the plan's {tile(base)}"
                    assert rec[tile(p)] <= BOUNDARY_COST * rec[tile(base)], (kind, shape, name, factor, rec)
                    moved.add((kind, shape, tile(p)))
    # the record holds nothing stale: every recorded alternative is one a perturbation reaches
    for (kind, shape), rec in RECORDED_BOUNDARIES.items():
        for t in list(rec)[1:]:
            assert (kind, shape, t) in moved, f"{kind} {shape}: recorded alternative {t} is no longer reached"


# (kind, shape, kernel that has to run, its time, the other's: wave-split tile against the kernel the constants table names,
# few workgroups against many), in microseconds as for RECORDED_BOUNDARIES; both sides of each line that tile_choice.h draws
MEASURED_CHOICES = [
    ("fp8", (16, 36864, 2304), "dma3", 19.3, 22.9), ("fp8", (16, 50688, 5120), "dma3", 51.3, 57.3), ("int8", (12, 17408, 1024), "dma3", 7.1, 9.0),
    # (rows 4096 bytes apart: the mid-M tile's K loops start at different blocks; the wave-split tile was the faster one, 29.5 against 31.7 and
    # 28.4 against 32.2, when they all started at the first)
    ("fp8", (16, 30464, 4096), "dma3", 23.5, 25.7), ("fp8_scaled", (16, 30464, 4096), "dma3", 23.9, 25.1),
    ("fp8", (1, 20736, 4096), "decode_wavesplit", 19.0, 24.4), ("fp8", (8, 20736, 4096), "decode_wavesplit", 21.3, 24.4),
    ("fp8", (6, 27392, 3584), "wavesplit_tile", 21.8, 23.6), ("int8", (11, 28672, 4096), "wavesplit_tile", 26.2, 29.8),
    ("fp8", (2616, 704, 10368), "dma3", 37.4, 53.2), ("fp8", (1610, 960, 10496), "dma3", 34.7, 44.7), ("fp8_scaled", (2595, 384, 7168), "dma3", 19.3, 22.3),
    ("fp8", (1608, 576, 7168), "wavesplit_tile", 20.3, 23.1),
    ("fp8", (71, 17920, 14592), ("dma3", 128, 256, 3), 62.6, 81.0), ("fp8_scaled", (103, 19072, 17664), ("dma3", 128, 256, 3), 77.2, 96.2),
    ("fp8_ue8m0", (65, 9792, 10624), ("dma3", 96, 128, 3), 28.7, 39.2),
]


@pytest.mark.parametrize("kind,shape,want,us,other", MEASURED_CHOICES)
def test_the_faster_kernel_runs(kind, shape, want, us, other):
    p = plan_for(kind, *shape)
    assert us < other and want in (p["kernel"], (p["kernel"], p["bm"], p["bn"], p["splits"])), p


# A large weight comes from memory: (kind, shape, tile and splits that run).  us of the linear, and of the tile that the other times name:
COLD_CHOICES = [
    ("fp8", (139, 7168, 18432), ("dma3", 160, 128, 4)),  # 45.9, 52.5
    ("fp8", (158, 16384, 16640), ("dma3", 160, 128, 2)),  # 77.7, 104.6
    ("fp8_ue8m0", (254, 12288, 12416), ("dma3", 128, 192, 2)),  # 58.9, 68.9
    ("fp8_scaled", (510, 16512, 3456), ("pingpong", 256, 256, 1)),  # 44.2, 51.9
    ("int8", (63, 29184, 2816), ("dma3", 64, 128, 1)),  # 20.6, 27.2
    ("fp8", (44, 14336, 4096), ("wavesplit_tile", 64, 64, 1)),  # 17.7, 21.3
    # what it leaves alone: two token tiles in a split plan that fills the chip, the 256 x 256 tile, smaller weights
    ("fp8_ue8m0", (72, 21120, 8320), ("dma3", 128, 256, 3)),  # 44.8, 46.3
    ("fp8_ue8m0", (2556, 7168, 7168), ("pingpong", 256, 256, 1)),  # 155.3, 159.0
    ("fp8", (1608, 576, 7168), ("wavesplit_tile", 64, 64, 1)),  # 20.3, 23.1
]


@pytest.mark.parametrize("kind,shape,want", COLD_CHOICES)
def test_large_weights_run_the_measured_tile(kind, shape, want):
    p = plan_for(kind, *shape)
    assert (p["kernel"], p["bm"], p["bn"], p["splits"]) == want, p


# Weights that the caches may still hold, where a K split loses its reduce launch again, with three weights in turn (first pair of us:
# unsplit, split) and from memory (second pair) or only with three in turn
REDUCE_NOT_EARNED = [
    ("int8", (143, 9216, 7168)),  # 21.8, 27.2; 30.2, 34.1
    ("fp8_scaled", (218, 6144, 7168)),  # 21.8, 28.1; 29.9, 30.2
    ("int8", (166, 8192, 8192)),  # 24.6, 30.0; 33.5, 34.9
    ("int8", (216, 7168, 9216)),  # 37.1, 39.0 with eight weights in turn
    ("fp8", (153, 9216, 7168)),  # 27.9, 29.4; 32.0, 34.0
]


@pytest.mark.parametrize("kind,shape", REDUCE_NOT_EARNED)
def test_no_split_that_its_reduce_costs_more_than_it_gains(kind, shape):
    assert plan_for(kind, *shape)["splits"] == 1, plan_for(kind, *shape)


# Up to 16 tokens on weights that are loaded as a stream: (linear, shape, kernel and channel tile that run).  us, and what ran otherwise:
STREAMED_CHOICES = [
    ("block", (16, 14336, 18432), "wavesplit_tile", 64),  # 47.9, 64.1
    ("block", (4, 14336, 8192), "wavesplit_tile", 64),  # 24.6, 36.7
    ("int8", (4, 36864, 7168), "dma3", 192),  # 44.2, 53.2
    ("token_fp8", (8, 24576, 7168), "wavesplit_tile", 32),  # 33.4, 39.7
    ("ue8m0", (1, 12288, 13312), "wavesplit_tile", 16),  # 30.3, 38.2
    # rows 4096 bytes apart too: the mid-M tile starts its K loops at different blocks there
    ("int8", (4, 28672, 4096), "dma3", 128),  # 24.2, 26.3
    ("token_fp8", (8, 28672, 4096), "dma3", 128),  # 24.1, 26.3
    # one and two tokens from the second turn of the register kernel on
    ("ue8m0", (1, 16384, 7552), "wavesplit_tile", 64),  # 21.9, 24.2
    # what stays: one turn of that kernel at one and two tokens, a tile that another models within 8 % of
    ("block", (1, 36864, 3584), "decode_wavesplit", 16),  # 23.3, 24.8
    ("int8", (2, 28672, 4096), "decode_wavesplit", 16),  # 23.5, 24.2
    ("int8", (2, 9728, 12672), "wavesplit_tile", 64),  # 25.6, 27.9
]


@pytest.mark.parametrize("kind,shape,kernel,bn", STREAMED_CHOICES)
def test_streamed_weights_run_the_measured_kernel(kind, shape, kernel, bn):
    from sglang_amd import _lib

    p = _lib.linear_plan(kind, *shape)
    assert (p["kernel"], p["bn"]) == (kernel, bn), p


# Small layers of short K at decode sizes: (linear, shape, kernel that runs).  us a call, and what ran otherwise:
SMALL_CHOICES = [
    ("ue8m0", (13, 5888, 1536), "wavesplit_tile"),  # 6.5, 8.1
    ("int8", (7, 1088, 1024), "wavesplit_tile"),  # 4.5, 5.3
    ("ue8m0", (7, 1600, 640), "wavesplit_tile"),  # 5.3, 8.4
    ("token_fp8", (16, 4288, 1280), "wavesplit_tile"),  # 6.8, 8.7
    ("block", (15, 1408, 1920), "wavesplit_tile"),  # 7.4, 11.7
    ("block", (16, 512, 512), "wavesplit_tile"),  # 4.2, 8.1
    ("ue8m0", (9, 128, 1024), "wavesplit_tile"),  # 4.1, 6.1
    ("token_fp8", (1, 2048, 128), "wavesplit_tile"),  # 3.3, 6.2
    # what stays: up to four tokens with K of 8 blocks and more (4.7, the tile no faster), many token values a workgroup, many channels
    ("block", (2, 2688, 1280), "decode_wavesplit"),  # 4.7, 4.8
    ("block", (16, 4096, 2048), "decode_wavesplit"),  # 5.8, 8.2
    ("ue8m0", (16, 16896, 640), "decode"),  # 8.3, 10.0
]


@pytest.mark.parametrize("kind,shape,kernel", SMALL_CHOICES)
def test_small_layers_run_the_measured_kernel(kind, shape, kernel):
    from sglang_amd import _lib

    assert _lib.linear_plan(kind, *shape)["kernel"] == kernel, _lib.linear_plan(kind, *shape)


# (tokens, channels, K) on both sides of the line from which the weight-in-registers kernel is taken; the times stand at choose_mid_tile
RESIDENT_CHOICES = [
    ("block", (368, 32768, 512), True), ("ue8m0", (1493, 7296, 768), True), ("token_fp8", (827, 24576, 768), True), ("int8", (577, 20496, 768), True),
    ("int8", (975, 65584, 768), True), ("int8", (1100, 65584, 768), True), ("block", (430, 24576, 512), False), ("block", (458, 16384, 512), False),
    ("block", (1544, 4096, 512), False), ("block", (849, 6144, 512), False), ("block", (784, 5184, 512), False), ("block", (40, 34944, 768), False),
    ("token_fp8", (624, 16384, 640), False), ("token_fp8", (180, 24576, 512), False), ("int8", (4088, 1856, 768), False),
]


@pytest.mark.parametrize("kind,shape,taken", RESIDENT_CHOICES)
def test_resident_kernel_is_taken_where_the_rule_says(kind, shape, taken):
    from sglang_amd import _lib

    assert (_lib.linear_plan(kind, *shape)["kernel"] == "resident") == taken, _lib.linear_plan(kind, *shape)


def test_captured_linears_quantize_their_tokens_when_eager():
    from sglang_amd import _lib

    for kind, shape, kernels in CAPTURED_LINEARS:
        assert _lib.linear_plan(kind, *shape)["quantizer"] == "fused", (kind, shape, kernels)


def test_every_route_constant_has_its_name():
    """The names follow the constants one by one: none is blank, and those at the end of each group still have their values."""
    from sglang_amd import _lib

    constants = _lib.route_constants()
    assert all(constants) and constants["limits.half_decode_min_kblocks"] == 24.0
    assert constants["limits.cold_margin"] == 0.92 and constants["streamed.tile"] == 1.55 and constants["quant.saved"] == 1.4


def test_perturbed_plan_query():
    import ctypes

    from sglang_amd import _lib

    L = _lib.lib()
    n = L.mi355_route_constant_count()
    assert n == len(_lib.route_constants()) > 150 and L.mi355_route_constant_name(n) is None and L.mi355_route_constant_name(-1) is None
    assert _lib.route_constants()["pp_fp8_us_per_kblock"] == 1.39
    buf = ctypes.create_string_buffer(256)
    assert L.mi355_gemm_plan_perturbed(1, 128, 7168, 18432, 1, n, 1.1, buf, len(buf)) == 1
    assert L.mi355_gemm_plan_perturbed(1, 128, 7168, 18432, 1, 0, 0.0, buf, len(buf)) == 1
    # a factor of one is the plain query, and the perturbed copy does not outlive its call
    for kind, shape in (("fp8", (128, 7168, 18432)), ("int8", (256, 4096, 14336)), ("fp8", (4096, 36864, 7168))):
        assert _lib.gemm_plan_perturbed(kind, *shape, 3, 1.0) == _lib.gemm_plan(kind, *shape)
    far = _lib.gemm_plan_perturbed("fp8", 256, 36864, 7168, list(_lib.route_constants()).index("scaled.pp_block"), 10.0)
    assert far["kernel"] == "dma3" and _lib.gemm_plan("fp8", 256, 36864, 7168)["kernel"] == "pingpong"  # ten times slower it loses


def test_plan_query_rejects_bad_arguments():
    import ctypes

    from sglang_amd import _lib

    L = _lib.lib()
    buf = ctypes.create_string_buffer(8)
    assert L.mi355_fp8_blockwise_mm_plan(16, 128, 128, 1, buf, len(buf)) == 1 and b"too small" in L.mi355_last_error()
    assert L.mi355_int8_scaled_mm_plan(0, 128, 128, 1, buf, len(buf)) == 1
    assert L.mi355_fp8_blockwise_mm_plan(16, 128, 128, 1, None, 0) == 1
    assert L.mi355_fp8_blockwise_mm_ue8m0_plan(16, 128, 128, 1, buf, len(buf)) == 1 and L.mi355_fp8_scaled_mm_plan(16, 0, 128, 1, buf, len(buf)) == 1
    p = _lib.gemm_plan("fp8", 13, 19584, 7168)
    assert p["kernel"] == "decode" and p["splits"] == 7
    p = _lib.gemm_plan("fp8", 13, 18432, 7168)
    assert (p["kernel"], p["bm"], p["bn"]) == ("wavesplit_tile", 16, 64)
    p = _lib.gemm_plan("fp8", 13, 36864, 7168)  # one round of unsplit 64 x 192 tiles beats the split streaming kernel
    assert (p["kernel"], p["bm"], p["bn"], p["splits"]) == ("dma3", 64, 192, 1)
    p = _lib.gemm_plan("fp8", 1, 36864, 7168)
    assert p["kernel"] == "decode_wavesplit" and p["splits"] == 1 and p["bn"] == 16
    p = _lib.gemm_plan("fp8", 3, 36864, 7168)  # two channel tiles per workgroup from three tokens on
    assert p["kernel"] == "decode_wavesplit" and p["bn"] == 32
    assert _lib.gemm_plan("fp8_ue8m0", 8, 32840, 3328)["exponents"] == "unpacked"  # (N % 16 != 0: the generic kernel or the tile, on fp32 scales)


def test_block_linear_plan():
    """The one-call linear quantizes inside the GEMM kernel - the wave-split kernels for few tokens, the mid-M kernel's producer
    waves where one round of unsplit tiles fills the chip, the streaming kernel's prologue - except where a quantizer launch in
    front of a wave-split kernel was measured faster, and beyond decode sizes."""
    import ctypes

    from sglang_amd import _lib

    for shape, want in (((1, 36864, 7168), ("fused", "dma3")), ((3, 36864, 7168), ("fused", "dma3")), ((8, 36864, 7168), ("fused", "dma3")),
                        ((1, 28672, 4096), ("fused", "decode_wavesplit")), ((8, 24576, 7168), ("fused", "dma3")), ((16, 512, 512), ("fused", "wavesplit_tile")), ((16, 16896, 512), ("fused", "decode")),
                        ((16, 2048, 7168), ("launch", "wavesplit_tile")), ((8, 7168, 2048), ("fused", "wavesplit_tile")), ((4, 7168, 2048), ("fused", "decode_wavesplit")),
                        ((4, 7168, 18432), ("launch", "wavesplit_tile")), ((16, 7168, 2048), ("fused", "wavesplit_tile")),
                        ((128, 7168, 2048), ("launch", "wavesplit_tile")), ((4, 1000, 1024), ("launch", "generic"))):
        p = _lib.block_linear_plan(*shape)
        assert (p["quantizer"], p["kernel"]) == want, (shape, p)
        if p["quantizer"] == "launch":
            assert {k: v for k, v in p.items() if k != "quantizer"} == _lib.gemm_plan("fp8", *shape)
    # where the one call multiplies with the GEMM entry point's kernel and tiling (any plan with a quantizer launch, and the
    # fused plans whose kernel the GEMM entry point takes too) the reference-named wrappers equal their two calls bit for bit
    from sglang_amd.fp8_utils import _one_call_takes_the_same_gemm

    for shape, want in (((8, 36864, 7168), True), ((16, 2048, 7168), True), ((4, 7168, 18432), True), ((4100, 1024, 256), True),
                        ((40, 200, 384), True), ((1, 28672, 4096), True), ((1, 36864, 7168), False), ((3, 36864, 7168), False), ((8, 24576, 7168), False)):
        assert _one_call_takes_the_same_gemm(*shape) == want, shape
    # the other linears promise that wherever they are: their GEMM is the one the entry point alone takes
    gemm = {"ue8m0": "fp8_ue8m0", "token_fp8": "fp8_scaled", "int8": "int8"}
    for shape in LINEAR_SHAPES:
        for kind in ("ue8m0", "token_fp8"):  # (INT8 sums are exact in any kernel)
            p, q = _lib.linear_plan(kind, *shape), _lib.gemm_plan(gemm[kind], *shape)
            assert all(p[k] == q[k] for k in p if k != "quantizer") or q.get("exponents") == "unpacked", (kind, shape, p, q)
    buf = ctypes.create_string_buffer(256)
    assert _lib.lib().mi355_fp8_block_linear_plan(4, 1024, 1000, buf, len(buf)) == 1  # K not a multiple of 128
    assert _lib.lib().mi355_fp8_block_linear_plan(4, 1024, 1024, buf, 8) == 1 and b"too small" in _lib.lib().mi355_last_error()


@pytest.mark.parametrize("kind,M,N,K", [("fp8", 16, 2048, 7168), ("fp8", 128, 36864, 7168), ("int8", 256, 4096, 14336)])
def test_workspace_covers_the_plan(kind, M, N, K):
    from sglang_amd import _lib

    L = _lib.lib()
    p = plan_for(kind, M, N, K)
    ws = (L.mi355_fp8_blockwise_mm_workspace_bytes if kind == "fp8" else L.mi355_int8_scaled_mm_workspace_bytes)(M, N, K)
    assert ws >= (p["splits"] * M * N * 4 if p["splits"] > 1 else 0)


GEMM_WORKSPACES = {"fp8": "mi355_fp8_blockwise_mm_workspace_bytes", "fp8_ue8m0": "mi355_fp8_blockwise_mm_ue8m0_workspace_bytes",
                   "fp8_scaled": "mi355_fp8_scaled_mm_workspace_bytes", "int8": "mi355_int8_scaled_mm_workspace_bytes"}


def test_workspace_covers_every_kind_asked_in_turn():
    """The size is kept for the shapes met last: it is each shape's and kind's own, whatever was asked before."""
    from sglang_amd import _lib

    L = _lib.lib()
    rng = random.Random(5)
    shapes = [(rng.choice((3, 9, 16, 17, 33, 48, 96, 160, 387, 1100)), 8 * rng.randint(2, 4000), 128 * rng.randint(1, 160)) for _ in range(600)]
    first = {}
    for _ in range(2):  # the second turn meets some sizes kept and some replaced
        for s in shapes:
            for kind, name in GEMM_WORKSPACES.items():
                size = getattr(L, name)(*s)
                p = _lib.gemm_plan(kind, *s)
                assert size >= (p["splits"] * s[0] * s[1] * 4 if p["splits"] > 1 else 0), (kind, s, p)
                assert first.setdefault((kind, s), size) == size, (kind, s)


def test_host_work_of_a_workspace_query():
    """In units of a query that returns at once (M = 0; some 0.5 us): a known shape is a look at the table, and a token count not met
    before works out the plans of the one kind asked for (measured 1 and 9 of these units; 6 and 35 where a query worked out
    every FP8 kind's plans each time)."""
    from sglang_amd import _lib

    ask = _lib.lib().mi355_fp8_block_linear_workspace_bytes
    K, N = 18432, 7168

    def cost(tokens):
        t = time.perf_counter()
        for M in tokens:
            ask(M, N, K)
        return (time.perf_counter() - t) / len(tokens)

    fresh = iter(range(20, 1420, 70))
    trials = [(cost([0] * 400), cost([200] * 400), cost(range(m := next(fresh), m + 70))) for _ in range(20)]
    nothing, known, new = (min(t) for t in zip(*trials))
    assert known < 2 * nothing, (nothing, known)
    assert new < 20 * nothing, (nothing, new)


def test_host_work_of_a_known_linear():
    """What a linear does is kept per shape: a query for a large weight at decode sizes, which takes the longest to work out, costs what
    any other known one does (1.0; 1.5 where it was worked out on every call)."""
    import ctypes

    from sglang_amd import _lib

    ask, buf = _lib.lib().mi355_fp8_block_linear_plan, ctypes.create_string_buffer(256)

    def cost(M, N, K):
        t = time.perf_counter()
        for _ in range(400):
            ask(M, N, K, buf, len(buf))
        return time.perf_counter() - t

    trials = [(cost(4096, 36864, 7168), cost(8, 36864, 7168), cost(16, 24576, 7168)) for _ in range(30)]
    any_other, *large = (min(t) for t in zip(*trials))
    assert max(large) < 1.25 * any_other, (any_other, large)


def test_grouped_plan_bounds_hold_for_any_routing():
    """The grouped GEMM sizes its tile tables and grids on the host from (experts, stacked rows) alone, while the real
    tile counts come from row counts that only exist on the device.  Replay the device rule here (256-row tiles; a rest of
    129..255 rows is one more; a rest of 1..128 rows becomes small tiles of the height the plan names; small tiles for every row
    where the plan has no 256-row launch) for random and adversarial routings: the host bounds must never be exceeded."""
    import random

    from sglang_amd import _lib

    rnd = random.Random(7)
    cases = []
    for _ in range(300):
        E = rnd.choice([1, 2, 3, 8, 16, 64, 256, 300])
        kind = rnd.choice(["uniform", "skewed", "tiny", "edges"])
        if kind == "uniform":
            sizes = [rnd.randint(0, 600) for _ in range(E)]
        elif kind == "skewed":
            sizes = [rnd.choice([0, 0, 1, 2, 5000]) for _ in range(E)]
        elif kind == "tiny":
            sizes = [rnd.randint(0, 3) for _ in range(E)]
        else:
            sizes = [rnd.choice([1, 63, 64, 65, 127, 128, 129, 255, 256, 257, 384, 385]) for _ in range(E)]
        cases.append(sizes)
    cases += [[128] * 256, [129] * 256, [1] * 256, [64] * 300, [65] * 300, [385] * 16, [0] * 8 + [1]]
    kernels = set()
    for sizes in cases:
        E, total = len(sizes), sum(sizes)
        if total == 0:
            continue
        for N, K in ((512, 1024), (4096, 7168)):
            plan = _lib.grouped_gemm_plan(E, total, N, K)
            bm = int(plan["small_tile"].split("x")[0])
            two_kinds = "pingpong" in plan["kernel"]
            kernels.add(plan["kernel"])
            big = small = 0
            for rows in sizes:
                b, rest = divmod(rows, 256) if two_kinds else (0, rows)
                if two_kinds and rest > 128:
                    b += 1
                else:
                    small += -(-rest // bm)
                big += b
            assert big <= plan["max_big_tiles"], (sizes[:8], big, plan)
            assert small <= plan["max_small_tiles"], (sizes[:8], small, plan)
        # the re-laid-out scale columns: expert e starts at align4(row0) + 4 e and is read in whole quads
        pitch = (total + 3) // 4 * 4 + 4 * E + 4
        row0 = 0
        for e, rows in enumerate(sizes):
            if rows:
                assert (row0 + 3) // 4 * 4 + 4 * e + (rows + 3) // 4 * 4 <= pitch
            row0 += rows
    assert len(kernels) == 3


@pytest.mark.parametrize("E,N,K", [(256, 512, 7168), (32, 4096, 7168), (64, 2048, 7168), (128, 1536, 2048)])
def test_grouped_plan_fetches_each_weight_once(E, N, K):
    """Calls bound by the stream of the experts' weights: experts of up to 128 rows get one token tile each (two of 64 rows
    fetch the weight twice: 32 experts of 128 rows, 7168 -> 4096, 254 against 208 us), and no 256-row launch stands in front where
    an expert has a few rows (256 of 4 rows: 174 against 172 us)."""
    from sglang_amd import _lib

    for rows in (1, 4, 16, 32):
        p = _lib.grouped_gemm_plan(E, E * rows, N, K)
        assert p["kernel"] == "grouped_dma3", (rows, p)
    for rows in (72, 96, 112, 128):
        p = _lib.grouped_gemm_plan(E, E * rows, N, K)
        assert p["small_tile"] == "128x256", (rows, p)


def test_mid_m_plans_are_consistent():
    """Whatever the time model picks, a split must give every K range some work and the ranges must cover K."""
    from sglang_amd import _lib

    for kind in ("fp8", "int8"):
        for M in (17, 32, 64, 65, 128, 129, 200, 256, 300, 512, 1000, 1024, 1025, 4096):
            for N, K in ((576, 7168), (1536, 7168), (7168, 18432), (36864, 7168), (6144, 4096), (4096, 14336), (256, 128), (512, 16384)):
                p = _lib.gemm_plan(kind, M, N, K)
                kb = -(-K // 128)
                assert p["splits"] >= 1 and p["kb_per_split"] >= 1
                assert p["kb_per_split"] * p["splits"] >= kb and p["kb_per_split"] * (p["splits"] - 1) < kb, (kind, M, N, K, p)
                if p["kernel"] == "dma3":  # the tile shapes that are compiled; splits need N % 4 == 0
                    assert p["bm"] in (64, 96, 128, 160, 192, 256) and p["bn"] in (128, 192, 256), (kind, M, N, K, p)
                    assert p["splits"] == 1 or N % 4 == 0
