// Grouped blockwise-scaled FP8 GEMM for gfx950: the expert GEMMs of a mixture-of-experts layer in one call.
//
// What the reference's fp8_blockwise_scaled_grouped_mm computes (sgl-kernel/csrc/moe/fp8_blockwise_moe_kernel.cu:650-810,
// per-expert operand addresses as in sgl-kernel/csrc/moe/cutlass_moe_helper.cu:37-69): token rows of all experts are
// stacked in one matrix a [total_m, K] with their 1 x 128 group scales [total_m, K / 128]; expert e owns the rows
// expert_offsets[e] .. + problem_sizes[e][0], multiplies them with its own weight b[e] [N, K] (128 x 128 block scales
// scales_b[e] [N / 128, K / 128]) and writes the same rows of out [total_m, N].  problem_sizes and expert_offsets live
// on the device (they come out of the routing kernel), so the tile schedule is built on the device too:
//   1. grouped_prepare_kernel - one workgroup turns the problem sizes, by prefix sums over the experts' tile counts, into one
//      record per token tile (expert, rows, position) in two tables, 256-row tiles and 64/128-row tiles, each headed by
//      its number of records; sizes are clamped into the stacked matrix, so inconsistent routing data cannot make a later kernel read
//      or write out of bounds.  The other workgroups re-lay the token scales out M-major (what the direct-to-LDS GEMMs read with
//      16-byte loads), every expert padded to start on a whole quad of rows; they find the experts of their 32 rows themselves and
//      wait for nobody (two launches, one after the other, took 9.6 us with the gap between them, this one 5);
//   2. fp8_grouped_pp_kernel (gemm_fp8_pp.hip), the two-phase 256 x 256 tile kernel, over the first table, then
//      fp8_grouped_dma_kernel (gemm_fp8_dma3.hip), the mid-M tile of 64 or 128 tokens x 128 or 256 channels, over the second:
//      one workgroup per (token tile, channel tile).  The first launch is left out when no expert can have more than
//      128 rows, and where small tiles alone model faster (grouped_run): then every row goes to the second table.
// Where the reference takes device arrays of per-expert pointers, strides and scale layouts as scratch that its own
// set-up kernel fills, this interface takes the base pointers and strides and keeps its scratch in the workspace.
#include "tile_choice.h"

namespace mi355 {
namespace {

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Tile heights.  An expert's rows are cut into 256-row tiles for the two-phase kernel; what is left (fewer than 256 rows)
// becomes one more 256-row tile when it is more than 128 rows, otherwise 64- or 128-row tiles for the three-stage kernel
// (one height per call, chosen on the host from the average rows per expert).  Measured on the dense kernels: per output
// element a 128-row tile costs 1.5x and a 64-row tile 2.3x of a 256-row tile when both are bound by the matrix pipe.
constexpr int BIG = 256;

struct ExpertTiles {
  int row0, rows, big, small, small_first;  // tiles of each kind; first row (inside the expert) of the small tiles
};
__device__ __forceinline__ ExpertTiles expert_tiles(const int32_t* problem_sizes, const int32_t* expert_offsets, int e, int E,
                                                    int total_m, int bm, bool use_big) {
  ExpertTiles t{0, 0, 0, 0, 0};
  if (e >= E) return t;
  t.row0 = min(max(expert_offsets[e], 0), total_m);
  t.rows = min(max(problem_sizes[3 * e], 0), total_m - t.row0);
  t.big = use_big ? t.rows / BIG : 0;
  const int rest = t.rows - t.big * BIG;
  if (use_big && rest > 128) t.big += 1;
  else t.small = (rest + bm - 1) / bm;
  t.small_first = t.big * BIG;
  return t;
}

struct GroupedTables {
  int E, total_m, bm, use_big, max_big, max_small;
  v4i *big_tiles, *small_tiles;
};
__device__ void grouped_plan(const int32_t* problem_sizes, const int32_t* expert_offsets, const GroupedTables& g) {
  const int E = g.E, bm = g.bm, max_big = g.max_big, max_small = g.max_small;
  v4i *big_tiles = g.big_tiles, *small_tiles = g.small_tiles;
  __shared__ int scan_b[256], scan_s[256];
  int base_b = 0, base_s = 0;
  for (int c = 0; c < E; c += 256) {
    const int e = c + (int)threadIdx.x;
    const ExpertTiles t = expert_tiles(problem_sizes, expert_offsets, e, E, g.total_m, bm, g.use_big);
    scan_b[threadIdx.x] = t.big, scan_s[threadIdx.x] = t.small;
    __syncthreads();
    for (int d = 1; d < 256; d <<= 1) {  // inclusive prefix sums
      const int vb = (int)threadIdx.x >= d ? scan_b[threadIdx.x - d] : 0;
      const int vs = (int)threadIdx.x >= d ? scan_s[threadIdx.x - d] : 0;
      __syncthreads();
      scan_b[threadIdx.x] += vb, scan_s[threadIdx.x] += vs;
      __syncthreads();
    }
    const int first_b = base_b + scan_b[threadIdx.x] - t.big, first_s = base_s + scan_s[threadIdx.x] - t.small;
    for (int j = 0; j < t.big; ++j)
      if (first_b + j < max_big) big_tiles[1 + first_b + j] = v4i{e, t.row0, t.rows, j * BIG};
    for (int j = 0; j < t.small; ++j)
      if (first_s + j < max_small) small_tiles[1 + first_s + j] = v4i{e, t.row0, t.rows, t.small_first + j * bm};
    base_b += scan_b[255], base_s += scan_s[255];
    __syncthreads();
  }
  // record 0 of each table: how many follow (consistent routing data never exceeds the bounds)
  if (threadIdx.x == 0) {
    big_tiles[0] = v4i{min(base_b, max_big), 0, 0, 0};
    small_tiles[0] = v4i{min(base_s, max_small), 0, 0, 0};
  }
}

// Workgroup (x, y) < (chunks, K blocks / 32): out[kb * pitch + col(e) + m] = sa[(row0 + m) * sa_sm + kb * sa_sk] for 32 stacked rows x 32
// K blocks, col(e) = ((row0 + 3) & ~3) + 4 * e, through LDS so that both sides are contiguous.  The last x: the tables.
constexpr int CHUNK = 32;
__global__ __launch_bounds__(256) void grouped_prepare_kernel(const int32_t* problem_sizes, const int32_t* expert_offsets, GroupedTables g,
                                                              const float* sa, int64_t sa_sm, int64_t sa_sk, float* out, int64_t pitch, int KB) {
  if (blockIdx.x == gridDim.x - 1) {
    if (blockIdx.y == 0) grouped_plan(problem_sizes, expert_offsets, g);
    return;
  }
  __shared__ float tile[32][CHUNK + 1];
  __shared__ int owners[CHUNK], column[CHUNK];  // per row of the chunk: how many experts of the batch own it, and the row's column
  const int r0 = blockIdx.x * CHUNK, r1 = min(r0 + CHUNK, g.total_m), k0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const bool k_fast = sa_sk < sa_sm;
#pragma unroll
  for (int i = ty; i < 32; i += 8) {
    const int m = k_fast ? i : tx, kb = k_fast ? tx : i;
    if (r0 + m < r1 && k0 + kb < KB) tile[kb][m] = sa[(int64_t)(r0 + m) * sa_sm + (int64_t)(k0 + kb) * sa_sk];
  }
  auto store = [&](int m, int col) {
    for (int kb = ty; kb < 32; kb += 8)
      if (k0 + kb < KB) out[(int64_t)(k0 + kb) * pitch + col] = tile[kb][m];
  };
  for (int c = 0; c < g.E; c += 256) {
    if (threadIdx.x < CHUNK) owners[threadIdx.x] = 0;
    __syncthreads();
    const int e = c + (int)threadIdx.x;
    const ExpertTiles t = expert_tiles(problem_sizes, expert_offsets, e, g.E, g.total_m, g.bm, false);
    const int lo = max(t.row0, r0), hi = min(t.row0 + t.rows, r1), shift = ((t.row0 + 3) & ~3) + 4 * e - t.row0;
    int shared_rows = 0;
    if (e < g.E)
      for (int m = lo; m < hi; ++m) shared_rows |= atomicAdd(&owners[m - r0], 1), column[m - r0] = shift + m;
    if (__syncthreads_or(shared_rows) == 0) {  // every row has one owner at most: all rows at once
      if (owners[tx]) store(tx, column[tx]);
    } else {  // inconsistent offsets: expert by expert
      for (int i = 0; i < 256 && c + i < g.E; ++i) {
        const ExpertTiles o = expert_tiles(problem_sizes, expert_offsets, c + i, g.E, g.total_m, g.bm, false);
        const int m = r0 + tx;
        if (m >= o.row0 && m < min(o.row0 + o.rows, r1)) store(tx, ((o.row0 + 3) & ~3) + 4 * (c + i) + m - o.row0);
      }
    }
    __syncthreads();
  }
}

struct GroupedPlan {
  int bm;                  // height of the small tiles
  int max_big, max_small;  // upper bounds on the number of tile records of each kind
  int64_t pitch;           // floats per K block in the re-laid-out token scales
  size_t big_bytes, scale_bytes;
};

GroupedPlan grouped_plan(int64_t E, int64_t total_m, int64_t K) {
  GroupedPlan pl;
  pl.bm = total_m > 64 * E ? 128 : 64;  // by the average rows per expert; the sizes themselves are on the device
  pl.max_big = (int)(total_m / 129);    // every 256-row tile covers more than 128 rows
  // an expert leaves at most 128 rows to small tiles, and every small tile covers at least one row
  pl.max_small = (int)std::min<int64_t>(total_m, E * (128 / pl.bm));
  // the last expert's column is at most align4(total_m) - rows + 4 (E - 1) + 3, and the GEMM reads whole quads up to
  // align4(rows) past it: one more quad of slack keeps that inside the row (and inside the workspace for the last row)
  pl.pitch = ((total_m + 3) & ~3ll) + 4 * E + 4;
  pl.big_bytes = align256((size_t)(pl.max_big + 1) * sizeof(v4i));  // record 0 holds the count
  pl.scale_bytes = align256((size_t)pl.pitch * (size_t)((K + KSTEP - 1) / KSTEP) * 4u);
  return pl;
}

// What runs: with or without the 256-row tiles, and the shape of the small ones.
struct GroupedRun {
  bool use_big;
  int bm, bn, max_big, max_small;
  bool few;  // at most a workgroup per CU is expected
};

size_t grouped_small_bytes(const GroupedRun& r) { return align256((size_t)(r.max_small + 1) * sizeof(v4i)); }

// Small tiles alone against 256-row tiles plus small ones, by the tile times of the dense GEMM for evenly spread rows; the second
// launch costs about 4 us, also when no expert fills a 256-row tile.  Measured (whole
// call, us, always with 256-row tiles / as chosen): 32 experts, 5392 rows, K = 896 -> N = 384 34.2 / 13.8;  8, 396, 1024 -> 1024
// 17.0 / 12.3;  64, 7112, 1408 -> 1792 78.7 / 62.9;  8, 26, 6144 -> 384 29.7 / 21.5.
GroupedRun grouped_run(int64_t E, int64_t total_m, int64_t N, int64_t K, const GroupedPlan& pl) {
  const TileTimes& t = SCALED_TIMES;
  const int64_t active = std::min(E, total_m), rows = ceil_div(total_m, active), kb = ceil_div(K, KSTEP);
  auto small_us = [&](int bm, int bn, int64_t tiles_m, int64_t* workgroups) {
    int i = 0;
    while (MID_TILES[i].bm != bm || MID_TILES[i].bn != bn) ++i;
    const int64_t wg = tiles_m * ceil_div(N, bn);
    const bool two = bm + bn == 192 && wg > NUM_CUS;
    if (workgroups) *workgroups = wg;
    return rounds_of(wg, two ? 2 * NUM_CUS : NUM_CUS, [&](double fill) { return t.tile[i] + (double)kb * t.block[i] * (two ? t.shared : 1.0) * (1.0 + t.busy * fill); });
  };
  // the weights of every active expert stream from memory once whatever the tiles
  const double stream = (double)active * (double)N * (double)K * 1e-6 / 5.0;
  const int64_t big = rows / BIG + (rows % BIG > 128), rest = rows % BIG > 128 ? 0 : rows % BIG;
  double best = std::max(small_us(pl.bm, 256, active * ceil_div(rest, pl.bm), nullptr) + rounds_of(active * big * ceil_div(N, 256), NUM_CUS, [&](double fill) {
                           return t.pp_tile + (double)kb * t.pp_block * (1.0 + t.pp_busy * fill);
                         }), stream) + (pl.max_big > 0 ? 4.0 : 0.0);
  GroupedRun r{pl.max_big > 0, pl.bm, 256, pl.max_big, pl.max_small, false};
  for (int bm = 64; bm <= 128; bm += 64)
    for (int bn = 256; bn >= 128; bn -= 128) {
      int64_t wg = 0;
      const double us = std::max(small_us(bm, bn, active * ceil_div(rows, bm), &wg), stream);
      if (us < 0.95 * best || us + 3.0 < best) {  // (bound by the weights' stream either way: the launch alone decides)
        best = us;
        r = GroupedRun{false, bm, bn, 0, (int)std::min<int64_t>(total_m, total_m / bm + E), wg <= NUM_CUS};
      }
    }
  return r;
}

}  // namespace
}  // namespace mi355

using namespace mi355;

extern "C" size_t mi355_fp8_blockwise_scaled_grouped_mm_workspace_bytes(int64_t num_experts, int64_t total_m, int64_t N,
                                                                        int64_t K) {
  if (num_experts <= 0 || total_m <= 0 || N <= 0 || K <= 0) return 0;
  const GroupedPlan pl = grouped_plan(num_experts, total_m, K);
  return pl.big_bytes + grouped_small_bytes(grouped_run(num_experts, total_m, N, K, pl)) + pl.scale_bytes;
}

extern "C" int mi355_fp8_blockwise_scaled_grouped_mm_plan(int64_t num_experts, int64_t total_m, int64_t N, int64_t K, char* buf,
                                                          size_t buf_len) {
  const char* what = "mi355_fp8_blockwise_scaled_grouped_mm_plan";
  clear_error();
  MI355_REQUIRE(buf && buf_len > 0, MI355_ERR_INVALID_ARGUMENT, "%s: no buffer", what);
  MI355_REQUIRE(num_experts > 0 && total_m > 0 && N > 0 && K > 0, MI355_ERR_INVALID_ARGUMENT, "%s: empty problem", what);
  const GroupedRun run = grouped_run(num_experts, total_m, N, K, grouped_plan(num_experts, total_m, K));
  const int n = snprintf(buf, buf_len, "kernel=%s small_tile=%dx%d max_big_tiles=%d max_small_tiles=%d tiles_n=%lld",
                         run.use_big ? "grouped_pingpong+grouped_dma3" : "grouped_dma3", run.bm, run.bn, run.max_big, run.max_small,
                         (long long)ceil_div(N, run.bn));
  MI355_REQUIRE(n > 0 && (size_t)n < buf_len, MI355_ERR_INVALID_ARGUMENT, "%s: buffer of %zu bytes is too small", what, buf_len);
  return MI355_OK;
}

extern "C" int mi355_fp8_blockwise_scaled_grouped_mm(const void* a, const void* b, const float* scales_a, const float* scales_b,
                                                     void* out, int out_dtype, const int32_t* problem_sizes,
                                                     const int32_t* expert_offsets, int64_t num_experts, int64_t total_m,
                                                     int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t b_expert_stride,
                                                     int64_t sa_sm, int64_t sa_sk, int64_t sb_expert_stride, int64_t sb_sn,
                                                     int64_t sb_sk, int64_t ldo, void* workspace, size_t workspace_bytes,
                                                     void* stream) {
  const char* what = "mi355_fp8_blockwise_scaled_grouped_mm";
  clear_error();
  MI355_REQUIRE(num_experts >= 0 && total_m >= 0 && N >= 0 && K >= 0, MI355_ERR_INVALID_ARGUMENT, "%s: negative shape", what);
  MI355_REQUIRE(out_dtype == MI355_BF16 || out_dtype == MI355_F16, MI355_ERR_INVALID_ARGUMENT,
                "%s: out_dtype must be bfloat16 or float16", what);
  if (num_experts == 0 || total_m == 0 || N == 0) return MI355_OK;
  MI355_REQUIRE(K > 0, MI355_ERR_INVALID_ARGUMENT, "%s: K must be positive", what);
  MI355_REQUIRE(a && b && scales_a && scales_b && out && problem_sizes && expert_offsets, MI355_ERR_INVALID_ARGUMENT,
                "%s: null pointer", what);
  MI355_REQUIRE(lda >= K && ldb >= K && ldo >= N, MI355_ERR_INVALID_ARGUMENT, "%s: row strides smaller than the row length", what);
  MI355_REQUIRE(K % KSTEP == 0, MI355_ERR_UNSUPPORTED, "%s: K must be a multiple of 128", what);
  MI355_REQUIRE(lda % 16 == 0 && ldb % 16 == 0 && b_expert_stride % 16 == 0 && (reinterpret_cast<uintptr_t>(a) & 15) == 0 &&
                    (reinterpret_cast<uintptr_t>(b) & 15) == 0,
                MI355_ERR_UNSUPPORTED, "%s: operand rows and expert strides must be 16-byte aligned", what);
  MI355_REQUIRE(num_experts < (1 << 24) && total_m < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31) &&
                    total_m * lda < (1ll << 32) && N * ldb < (1ll << 32),
                MI355_ERR_INVALID_ARGUMENT, "%s: dimensions out of range (row offsets must stay below 4 GiB)", what);
  const GroupedPlan pl = grouped_plan(num_experts, total_m, K);
  const GroupedRun run = grouped_run(num_experts, total_m, N, K, pl);
  const size_t small_bytes = grouped_small_bytes(run);
  MI355_REQUIRE(((int64_t)run.max_big + run.max_small) * ((N + run.bn - 1) / run.bn) < (1ll << 31), MI355_ERR_INVALID_ARGUMENT,
                "%s: too many tiles", what);
  const size_t need = pl.big_bytes + small_bytes + pl.scale_bytes;
  MI355_REQUIRE(workspace && workspace_bytes >= need, MI355_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", what,
                need, workspace_bytes);
  MI355_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, MI355_ERR_INVALID_ARGUMENT,
                "%s: workspace must be 256-byte aligned", what);

  hipStream_t st = static_cast<hipStream_t>(stream);
  uint8_t* wsp = static_cast<uint8_t*>(workspace);
  v4i* big_tiles = reinterpret_cast<v4i*>(wsp);
  v4i* small_tiles = reinterpret_cast<v4i*>(wsp + pl.big_bytes);
  float* sa_mm = reinterpret_cast<float*>(wsp + pl.big_bytes + small_bytes);
  const int KB = (int)(K / KSTEP);
  const GroupedTables tables{(int)num_experts, (int)total_m, run.bm, (int)run.use_big, run.max_big, run.max_small, big_tiles, small_tiles};
  hipLaunchKernelGGL(grouped_prepare_kernel, dim3((unsigned)((total_m + CHUNK - 1) / CHUNK + 1), (unsigned)((KB + 31) / 32)), dim3(256), 0, st,
                     problem_sizes, expert_offsets, tables, scales_a, sa_sm, sa_sk, sa_mm, pl.pitch, KB);
  int rc = check_launch(what);
  if (rc != MI355_OK) return rc;

  GroupedParams gp{};
  gp.g.a = static_cast<const uint8_t*>(a);
  gp.g.b = static_cast<const uint8_t*>(b);
  gp.g.sa = sa_mm, gp.g.sb = scales_b, gp.g.out = out;
  gp.g.M = 0, gp.g.N = (int)N, gp.g.K = (int)K;
  gp.g.lda = lda, gp.g.ldb = ldb, gp.g.ldo = ldo;
  gp.g.sa_sm = 1, gp.g.sa_sk = pl.pitch, gp.g.sb_sn = sb_sn, gp.g.sb_sk = sb_sk;
  gp.g.kb_total = KB;
  gp.g.out_dtype = out_dtype;
  gp.b_expert_stride = b_expert_stride;
  gp.sb_expert_stride = sb_expert_stride;
  gp.out_elem = 2;
  if (run.use_big) {
    gp.tiles = big_tiles, gp.max_tiles_m = run.max_big;
    rc = launch_fp8_grouped_pp(gp, st, what);
    if (rc != MI355_OK) return rc;
  }
  gp.tiles = small_tiles, gp.max_tiles_m = run.max_small;
  return launch_fp8_grouped_dma3(gp, run.bm, run.bn, run.few, st, what);
}
