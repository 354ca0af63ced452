// Which tile a GEMM runs on, by modelled time: the mid-M tiles (gemm_dma_tile.h) with or without split K, the small wave-split
// tiles (gemm_wavesplit_tile.h) and the 256 x 256 two-phase tile, next to what the route of the constants table names.
//
// The model was fitted to 60 000 timings of forced tiles (14 to 37 layers of K = 256 .. 18432 by N = 192 .. 36864, 1 to 4096
// tokens, all tiles and splits, weights rotated out of the caches, and results too where they are large): 4 % root mean square for
// the mid-M tiles, 6 % for the wave-split ones.  With larger operands than those shapes had, the wave-split tiles take 1.1 to 1.5
// times the modelled time: the limits below lie where they stop being the faster ones.
// The route that runs against the constants table alone, 720 random shapes (profiles/tile_choice_random_shapes.txt): 19 % faster for
// FP8, 21 % with packed exponents, 17 % per token, 22 % for INT8 (geometric means); more than 5 % slower at 13 shapes, by up to 17 %.
#pragma once

#include <algorithm>
#include <cmath>

#include "gemm_common.h"

namespace mi355 {

struct TileTimes {
  // mid-M tile: launch + rounds of one workgroup per CU (64 x 128: two where there are more workgroups than CUs, each then
  // `shared` times slower per block), each tile[i] + K blocks * block[i] * (1 + busy * fill); against the stream of both
  // operands at `stream` TB/s plus the result; a split adds its launch and its partial sums
  double launch, busy, split_us, split_us_per_mb, stream, stream_us, shared, result_us_per_mb;
  double tile[13], block[13];  // in the order of MID_TILES
  double pp_tile, pp_block, pp_busy, pp_store;  // 256 x 256; pp_store: a full round's result on its way to memory
  // wave-split tile: rounds of ws_tile + KB of operands * (ws_kb + ws_kb_busy * fill) + kilo-elements of the tile * ws_result,
  // together with the weight stream (ws_norm: how far the two overlap)
  double ws_launch, ws_tile, ws_kb, ws_kb_busy, ws_stream, ws_stream_us, ws_result, ws_norm;
  // weight in registers (gemm_resident.h): rounds of rs_tile + K blocks * rs_tile_block + steps * (rs_step + K blocks * rs_step_block) *
  // (1 + rs_busy * fill), a step being 64 tokens (steps of 32 count half)
  double rs_launch, rs_tile, rs_tile_block, rs_step, rs_step_block, rs_busy;
  // a weight that comes from memory (choose_cold_tile): a K block of a mid-M tile takes no less than cold + channels * cold_channel +
  // tokens * cold_token (64 x 128, two workgroups per CU: times cold_shared); its stream, of which every further token tile fetches
  // the share cold_again once more; K / 1000 * (channels * cold_ws_channel + tokens * cold_ws_token) for a wave-split tile and its stream
  // at cold_ws_stream times the rate above; 256 x 256: factors and busy of pp_block
  double cold, cold_channel, cold_token, cold_shared, cold_stream, cold_stream_us, cold_again, cold_split_us, cold_split_us_per_mb;
  double cold_ws_channel, cold_ws_token, cold_ws_stream, cold_ws_stream_us, cold_ws_norm;
  double cold_pp_tile, cold_pp_block, cold_pp_busy;
  double cold_cached;  // how much slower a tile may model by the times above, on weights that the caches may hold
};
// Up to 16 tokens, a weight loaded as a stream (choose_streamed_tile): rounds of `tile` + K / 1000 * (channels * channel + tokens * token) and
// the stream for the 16-token wave-split tiles; rounds of K blocks * (block + channels * block_channel + tokens * block_token), 64 x 128
// in two workgroups per CU `shared` times, and the stream for the unsplit mid-M tiles of 64 tokens.
struct StreamedTimes {
  double tile = 1.55, channel = 0.0201, token = 0.0103, stream = 8.70, stream_us = 3.02, norm = 2.06;
  double launch = 3.0, block = 0.098, block_channel = 0.00236, block_token = 0.00264, shared = 2.0, mid_stream = 7.06, mid_stream_us = 3.32;
};
// More than 16 tokens quantized inside the wave-split tile (choose_quant_tile), one round of workgroups: launch + tile + pieces of eight values a
// thread * piece (by GemmKind) + KB of weight * kb * (1 + kb_busy * fill) + kilo-elements of the tile * result.  `saved`: what the quantizer's
// launch takes beside the wave-split tile's modelled time; `many`: see there.
struct QuantTimes {
  double launch = 1.29, tile = 1.32, piece[4] = {0.310, 0.295, 0.370, 0.377}, many = 0.55, kb = 0.0051, kb_busy = 2.54, result = 0.488, saved = 1.4;
};
constexpr TileTimes SCALED_TIMES = {  // FP8 with scales in the K loop
    1.93, 0.586, 4.31, 0.217, 4.18, -4.54, 1.808, 0.421,
    {2.33, 2.83, 3.02, 3.40, 3.53, 4.64, 2.57, 3.31, 3.96, 4.32, 2.64, 3.53, 4.44},
    {0.219, 0.277, 0.317, 0.385, 0.419, 0.533, 0.288, 0.363, 0.441, 0.532, 0.334, 0.445, 0.535},
    7.88, 0.567, 1.70, 12.5,
    2.74, 1.041, 0.00591, 0.00334, 5.49, -3.81, 0.253, 1.511,
    3.63, 0.11, 0.406, 0.596, 0.186, 0.733,
    0.101, 0.0019, 0.0020, 1.42, 4.88, -0.45, 0.202, 3.27, 0.320,
    0.01269, 0.01362, 1.434, -1.44, 1.283,
    6.52, 1.774, 0.55, 1.08};
constexpr TileTimes PLAIN_TIMES = {  // FP8 with epilogue scales, INT8
    1.77, 0.777, 3.81, 0.251, 4.55, -2.24, 1.871, 0.402,
    {2.21, 2.72, 3.03, 3.17, 3.76, 4.72, 2.48, 3.12, 3.83, 4.14, 2.81, 3.80, 4.64},
    {0.165, 0.205, 0.240, 0.295, 0.333, 0.432, 0.224, 0.271, 0.339, 0.420, 0.278, 0.347, 0.431},
    8.48, 0.511, 1.70, 10.8,
    2.71, 1.017, 0.00609, 0.00343, 5.07, -4.41, 0.282, 1.673,
    3.64, 0.01, 0.435, 0.760, 0.217, 0.531,
    0.092, 0.0020, 0.0018, 1.37, 5.02, 1.55, 0.230, 3.16, 0.331,
    0.01247, 0.01387, 1.394, -1.13, 1.215,
    6.35, 1.730, 0.681, 1.03};
static_assert(sizeof(MID_TILES) / sizeof(MID_TILES[0]) == 13, "the tables above follow MID_TILES");

// Where the model is not asked or not trusted; both sides of each line stand beside the function that uses it.
struct TileLimits {
  double margin = 0.95, two_phase_margin = 0.90, large_weight_margin = 0.85, large_weight_max_tokens = 64.0;
  double mid_wavesplit_max_weight = 100e6, ragged_max_weight = 100e6, ragged_max_factor = 2.0;
  double ragged_min_kblocks = 2.0, ragged_two_phase_kblocks = 32.0, ragged_min_workgroups = 0.5 * NUM_CUS;
  double wavesplit_max_tokens_bytes = 16e6, wavesplit_long_k = 9216.0, wavesplit_long_k_max_tokens_bytes = 10e6, few_workgroups_max_tokens = 128.0;
  double decode_min_kblocks = 16.0, decode_padded_max_weight = 400e6, decode_max_weight = 140e6, decode_few_tokens_max_weight = 100e6;
  double decode_one_turn_min_kblocks = 30.0, decode_one_turn_kblocks = 32.0, decode_one_turn_max_channels = 16384.0, decode_one_turn_max_tokens = 10.0;
  double decode_few_tokens_f32 = 6.0, decode_few_tokens = 8.0, decode_long_kblocks = 64.0;
  double decode_short_min_kblocks = 8.0, decode_short_min_channels = 7168.0, decode_short_max_weight = 20e6, decode_short_min_tokens = 8.0;
  double resident_margin = 0.93, resident_rounds_margin = 0.95;
  double streamed_min_weight = 100e6, streamed_two_tokens_min_kblocks = 33.0;
  double small_min_tokens = 4.0, small_max_channels = 64.0 * NUM_CUS, small_max_tokens_values = 20800.0;
  double half_decode_min_kblocks = 24.0;
  double cold_min_weight = 40e6, cold_only_min_weight = 80e6, cold_margin = 0.92, cold_full_max_tokens = 128.0, cold_full_workgroups = 0.875 * NUM_CUS;
};
struct TileModel {
  TileTimes scaled = SCALED_TIMES, plain = PLAIN_TIMES;
  TileLimits limits;
  StreamedTimes streamed;
  QuantTimes quant;
};
constexpr int TILE_CONSTANT_COUNT = sizeof(TileModel) / sizeof(double);
// What the calling thread's dispatcher uses: the defaults above, or the perturbed copy a plan query installed.
const TileModel& tile_model();

namespace {

enum GemmKind { GK_F32, GK_UE8M0, GK_UNIT, GK_INT8 };  // FP8 with block scales, with exponents, with epilogue scales; INT8
enum TileFamily { TF_NONE, TF_DMA, TF_WAVESPLIT, TF_TWO_PHASE, TF_RESIDENT };

struct TileChoice {
  int family, bm, bn, splits;
  double us;
  int ranges = 0;  // TF_RESIDENT: workgroups that share a slice of channels
};

const TileTimes& tile_times(GemmKind kind) { return kind == GK_F32 || kind == GK_UE8M0 ? tile_model().scaled : tile_model().plain; }

double norm_of(double a, double b, double n) {
  if (b <= 0.1) return a;
  if (n != 6.0) return std::pow(std::pow(a, n) + std::pow(b, n), 1.0 / n);
  const double x = a * a * a, y = b * b * b;  // (most of a sweep's powers)
  return std::cbrt(std::sqrt(x * x + y * y));
}
// full rounds of `slots` workgroups and a partly filled one
template <class Round>
double rounds_of(int64_t workgroups, int64_t slots, Round round) {
  const int64_t full = workgroups / slots, rest = workgroups % slots;
  return (double)full * round(1.0) + (rest ? round((double)rest / (double)slots) : 0.0);
}

// (`most`: a time from which on the result does not matter; the powers are left out where the larger of the two bounds reaches it)
double dma_tile_us(const TileTimes& t, int i, int64_t M, int64_t N, int64_t K, int splits, double most = 1e30) {
  const int bm = MID_TILES[i].bm, bn = MID_TILES[i].bn;
  const double mn = (double)M * (double)N * 1e-6;
  const double stream = ((double)N + (double)M) * (double)K * 1e-6 / t.stream + mn * 2.0 * t.result_us_per_mb + t.stream_us;
  const double split = splits > 1 ? t.split_us + t.split_us_per_mb * splits * mn * 4.0 : 0.0;
  if (stream + split >= most) return most;
  const int64_t kb = ceil_div(K, KSTEP), wg = ceil_div(M, bm) * ceil_div(N, bn) * splits;
  const double blocks = (double)ceil_div(kb, splits);
  const bool two = bm + bn == 192 && wg > NUM_CUS;
  const double us = t.launch + rounds_of(wg, two ? 2 * NUM_CUS : NUM_CUS, [&](double fill) {
                      return t.tile[i] + blocks * t.block[i] * (two ? t.shared : 1.0) * (1.0 + t.busy * fill);
                    });
  return us + split >= most ? most : norm_of(us, stream, 6.0) + split;
}
double two_phase_us(const TileTimes& t, int64_t M, int64_t N, int64_t K) {
  const double blocks = (double)ceil_div(K, KSTEP);
  return t.launch + rounds_of(ceil_div(M, 256) * ceil_div(N, 256), NUM_CUS, [&](double fill) {
           return norm_of(t.pp_tile + blocks * t.pp_block * (1.0 + t.pp_busy * fill), t.pp_store * fill, 6.0);
         });
}
double wavesplit_tile_us(const TileTimes& t, int i, int64_t M, int64_t N, int64_t K, double most = 1e30) {
  const int bm = WAVESPLIT_TILES[i].bm, bn = WAVESPLIT_TILES[i].bn;
  const double kbytes = (double)(bm + bn) * (double)K * 1e-3;
  const double us = t.ws_launch + rounds_of(ceil_div(M, bm) * ceil_div(N, bn), NUM_CUS, [&](double fill) {
                      return t.ws_tile + kbytes * (t.ws_kb + t.ws_kb_busy * fill) + (double)(bm * bn) / 1024.0 * t.ws_result;
                    });
  const double stream = (double)N * (double)K * 1e-6 / t.ws_stream + t.ws_stream_us;
  return std::max(us, stream) >= most ? most : norm_of(us, stream, t.ws_norm);
}

// The tile of least time below `most`, or TF_NONE; us(i, most) and us(i, splits, most) time the i-th one.
template <class Time>
TileChoice fastest_wavesplit_tile(Time us, double most = 1e30) {
  TileChoice best{TF_NONE, 0, 0, 1, most};
  for (int i = 0; i < WAVESPLIT_MODELLED; ++i) {
    const double u = us(i, best.us);
    if (u < best.us) best = {TF_WAVESPLIT, WAVESPLIT_TILES[i].bm, WAVESPLIT_TILES[i].bn, 1, u};
  }
  return best;
}
template <class Time>
TileChoice fastest_dma_tile(int64_t M, int64_t N, int64_t K, Time us, double most = 1e30) {
  TileChoice best{TF_NONE, 0, 0, 1, most};
  const int64_t kb = ceil_div(K, KSTEP);
  for (int i = 0; i < 13; ++i) {
    const int64_t tiles = ceil_div(M, MID_TILES[i].bm) * ceil_div(N, MID_TILES[i].bn);
    int previous = 0;
    for (int want = 1; want <= 16; ++want) {
      const int per = (int)ceil_div(kb, want), splits = (int)ceil_div(kb, per);
      if (splits > 1 && (N % 4 != 0 || per < 4 || tiles * splits > 560 || tiles > 200)) break;
      if (splits == previous) continue;
      previous = splits;
      const double u = us(i, splits, best.us);
      if (u < best.us) best = {TF_DMA, MID_TILES[i].bm, MID_TILES[i].bn, splits, u};
    }
  }
  return best;
}
TileChoice best_wavesplit_tile(const TileTimes& t, int64_t M, int64_t N, int64_t K) {
  return fastest_wavesplit_tile([&](int i, double most) { return wavesplit_tile_us(t, i, M, N, K, most); });
}
TileChoice best_dma_tile(const TileTimes& t, int64_t M, int64_t N, int64_t K) {
  return fastest_dma_tile(M, N, K, [&](int i, int splits, double most) { return dma_tile_us(t, i, M, N, K, splits, most); });
}

// The same tiles with a weight that comes from memory.
double cold_dma_tile_us(const TileTimes& t, int i, int64_t M, int64_t N, int64_t K, int splits, double most = 1e30) {
  const int bm = MID_TILES[i].bm, bn = MID_TILES[i].bn;
  const int64_t tiles_m = ceil_div(M, bm), wg = tiles_m * ceil_div(N, bn) * splits;
  const double mn = (double)M * (double)N * 1e-6, fetches = 1.0 + t.cold_again * (double)(tiles_m - 1);
  const double stream = ((double)N * fetches + (double)M) * (double)K * 1e-6 / t.cold_stream + mn * 2.0 * t.result_us_per_mb + t.cold_stream_us;
  const double split = splits > 1 ? t.cold_split_us + t.cold_split_us_per_mb * splits * mn * 4.0 : 0.0;
  if (stream + split >= most) return most;
  const double blocks = (double)ceil_div(ceil_div(K, KSTEP), splits);
  const bool two = bm + bn == 192 && wg > NUM_CUS;
  const double fetch = (t.cold + t.cold_channel * bn + t.cold_token * (double)M / (double)tiles_m) * (two ? t.cold_shared : 1.0);
  const auto rounds = [&](auto larger) {
    return t.launch + rounds_of(wg, two ? 2 * NUM_CUS : NUM_CUS, [&](double fill) {
             return t.tile[i] + blocks * larger(t.block[i] * (two ? t.shared : 1.0) * (1.0 + t.busy * fill), fetch);
           });
  };
  if (rounds([](double x, double y) { return std::max(x, y); }) + split >= most) return most;
  return norm_of(rounds([](double x, double y) { return norm_of(x, y, 6.0); }), stream, 6.0) + split;
}
double cold_wavesplit_tile_us(const TileTimes& t, int i, int64_t M, int64_t N, int64_t K, double most = 1e30) {
  const int bm = WAVESPLIT_TILES[i].bm, bn = WAVESPLIT_TILES[i].bn;
  const int64_t tiles_m = ceil_div(M, bm);
  const double us = t.ws_launch + (double)ceil_div(tiles_m * ceil_div(N, bn), NUM_CUS) *
                                      (t.ws_tile + (double)K * 1e-3 * (t.cold_ws_channel * bn + t.cold_ws_token * (double)M / (double)tiles_m) +
                                       (double)(bm * bn) / 1024.0 * t.ws_result);
  const double stream = (double)N * (double)K * 1e-6 / (t.cold_stream * t.cold_ws_stream) + t.cold_ws_stream_us;
  return std::max(us, stream) >= most ? most : norm_of(us, stream, t.cold_ws_norm);
}
double cold_two_phase_us(const TileTimes& t, int64_t M, int64_t N, int64_t K) {
  const double blocks = (double)ceil_div(K, KSTEP);
  return t.launch + rounds_of(ceil_div(M, 256) * ceil_div(N, 256), NUM_CUS, [&](double fill) {
           return norm_of(t.cold_pp_tile + blocks * t.pp_block * t.cold_pp_block * (1.0 + t.cold_pp_busy * fill), t.pp_store * fill, 6.0);
         });
}

double resident_us(const TileTimes& t, int64_t M, int64_t N, int64_t K, int64_t step, int64_t ranges) {
  const int64_t kb = K / KSTEP, all = ceil_div(M, step), steps = ceil_div(all, ranges);
  const double halves = (double)(steps * step) / 64.0;
  return t.rs_launch + rounds_of(ceil_div(N, RESIDENT_CHANNELS) * ceil_div(all, steps), NUM_CUS, [&](double fill) {
           return t.rs_tile + (double)kb * t.rs_tile_block + halves * (t.rs_step + (double)kb * t.rs_step_block) * (1.0 + t.rs_busy * fill);
         });
}
// As many ranges of tokens as fill one, two or three rounds of workgroups, whichever models fastest; more rounds, each of which loads the
// weight again, only for 5 % (linears that this line moves to fewer: 0.96; packed exponents of K = 512, 1400 tokens -> 25576 two rounds
// 32.1 us, one 29.9).
TileChoice best_resident(GemmKind kind, int64_t M, int64_t N, int64_t K) {
  const TileTimes& t = tile_times(kind);
  TileChoice best{TF_NONE, 0, 0, 1, 1e30};
  if (K % KSTEP != 0 || K < 2 * KSTEP || K > RESIDENT_MAX_KBLOCKS * KSTEP || N % 8 != 0) return best;
  const int step = 2 * resident_half_step(kind == GK_UE8M0, (int)(K / KSTEP));
  const int64_t slices = ceil_div(N, RESIDENT_CHANNELS), most = ceil_div(M, step);
  double least = 1e30;
  for (int rounds = 1; rounds <= 3; ++rounds) {
    const int64_t ranges = std::min(std::max<int64_t>(rounds * NUM_CUS / slices, 1), most);
    const double us = resident_us(t, M, N, K, step, ranges);
    least = std::min(least, us);
    if (us < (rounds > 1 ? tile_model().limits.resident_rounds_margin : 1.0) * best.us) best = {TF_RESIDENT, step, RESIDENT_CHANNELS, 1, us, (int)ranges};
  }
  if (best.family != TF_NONE) best.us = least;
  return best;
}

// A linear of more than 16 tokens whose GEMM runs on the wave-split tile: the tile, of any size (all of them add the same products in the same
// order), that quantizes its tokens itself in the one launch, or TF_NONE.  Every channel tile repeats the quantizer's work, so it pays
// for layers of short K, as long as one round of workgroups does it (a second one never: 42 tokens 1536 -> 12288 16.3 us, two launches
// 10.3), and where the tile's tokens are at most ten pieces of eight values a thread.
// Fitted to 1600 timings of 320 linears: 6 % root mean square, the tile it names within 0.2 % of the best on average; `many` is what 16-token tiles
// take beyond four pieces, in the kernel of ten, by 160 more.  240 linears where one launch models no slower, one launch / two: 0.82 of the
// time in a graph (at most 1.04, but for two of 1.06 and 1.18), 0.64 eager; us in a graph, two launches / this: 18 tokens 512 -> 896 5.0 / 3.5,
// 669 tokens packed exponents 640 -> 384 6.8 / 4.3, 69 tokens per-token FP8 768 -> 384 5.3 / 4.2, INT8 103 tokens 768 -> 768 5.6 / 4.35.
// `eager_only`: with `many` it takes more of the GPU's time than two launches, less than the 2.4 us that a launch takes on the host; not in a
// capture, where they are not spent.  19 such linears 1.06 (0.94 to 1.23) of the two launches' time in a graph, 0.70 eager; graph, eager:
// 173 tokens packed exponents 2048 -> 256 5.5 / 6.7, 9.5 / 6.7; 48 tokens 2048 -> 768 5.8 / 6.6, 8.8 / 6.6; INT8 121 tokens 1536 -> 384 5.6 / 6.5, 8.9 / 6.4.
TileChoice choose_quant_tile(GemmKind kind, int64_t M, int64_t N, int64_t K, int plain_bm, int plain_bn, bool& eager_only) {
  const QuantTimes& q = tile_model().quant;
  double two_launches = 0.0;
  for (int i = 0; i < WAVESPLIT_MODELLED; ++i)
    if (WAVESPLIT_TILES[i].bm == plain_bm && WAVESPLIT_TILES[i].bn == plain_bn) two_launches = wavesplit_tile_us(tile_times(kind), i, M, N, K) + q.saved;
  TileChoice best{TF_NONE, 0, 0, 1, two_launches};
  eager_only = false;
  for (int i = 0; i < WAVESPLIT_QUANT_MODELLED; ++i) {
    const TileSize& t = WAVESPLIT_QUANT_TILES[i];
    const int64_t values = std::min<int64_t>(M, t.bm) * K, wg = ceil_div(M, t.bm) * ceil_div(N, t.bn);
    if (values > WAVESPLIT_QUANT_VALUES || wg > NUM_CUS) continue;
    const int64_t pieces = ceil_div(values, WAVESPLIT_QUANT_VALUES / 10);
    const double us = q.launch + q.tile + (double)pieces * q.piece[kind] + (double)(t.bn * K) * 1e-3 * q.kb * (1.0 + q.kb_busy * (double)wg / NUM_CUS) +
                      (double)(t.bm * t.bn) / 1024.0 * q.result;
    if (us >= best.us) continue;
    best = {TF_WAVESPLIT, t.bm, t.bn, 1, us};
    eager_only = t.bm == 16 && pieces > 4 && us + q.many >= two_launches;
  }
  return best;
}

// The wave-split tile: a large weight streams better through the wide tiles (K = 4096 -> N = 28672 at 48 tokens 27.2 against
// 33.6 us), and so does a large token matrix, which leaves the XCDs' L2s and is fetched again by every channel tile (mid-M / wave-split:
// K = 10368 -> N = 704 at 2616 tokens 37.4 / 53.2, 10496 -> 960 at 1610 34.7 / 44.7, per-token FP8 7168 -> 384 at 2595 19.3 / 22.3;
// but 7168 -> 576 at 1608 23.1 / 20.3).
bool wavesplit_allowed(int64_t M, int64_t N, int64_t K) {
  const TileLimits& l = tile_model().limits;
  const double token_bytes = (double)(M * K);
  return (double)(N * K) <= l.mid_wavesplit_max_weight && token_bytes <= l.wavesplit_max_tokens_bytes &&
         ((double)K <= l.wavesplit_long_k || token_bytes <= l.wavesplit_long_k_max_tokens_bytes);
}

// More than 16 tokens, K % 128 == 0, aligned operands: the fastest tile, or TF_NONE where `base`, what the route names (a mid-M
// tile or the two-phase tile), models within 5 % of it (the two-phase tile 10 %): below that the model does not order two tiles.
TileChoice choose_swept_tile(GemmKind kind, int64_t M, int64_t N, int64_t K, const TileChoice& base, double& base_us) {
  const TileTimes& t = tile_times(kind);
  TileChoice best = best_dma_tile(t, M, N, K);
  const TileLimits& l = tile_model().limits;
  if (wavesplit_allowed(M, N, K)) {
    const TileChoice ws = best_wavesplit_tile(t, M, N, K);
    if (ws.us < best.us) best = ws;
  }
  if (M > 128) {
    const double us = two_phase_us(t, M, N, K);
    if (us < best.us) best = {TF_TWO_PHASE, 256, 256, 1, us};
  }
  base_us = 1e30;
  if (base.family == TF_TWO_PHASE) base_us = two_phase_us(t, M, N, K);
  if (base.family == TF_DMA)
    for (int i = 0; i < 13; ++i)
      if (MID_TILES[i].bm == base.bm && MID_TILES[i].bn == base.bn) base_us = dma_tile_us(t, i, M, N, K, base.splits);
  // Bound by a large weight's stream, the model knows little of how many CUs it takes: K = 10880 -> N = 16896 at 36 tokens, 132
  // unsplit tiles instead of 198 split ones, 54.8 against 48.3 us.  From 65 tokens on the tile with more workgroups wins (14592 ->
  // 17920 at 71 tokens, 140 / 210 workgroups 81.0 / 62.6; per-token FP8 17664 -> 19072 at 103, 149 / 225, 96 / 77; but 10624 -> 9792 at
  // 65, 231 / 154, 28.7 / 39.2): of 24 shapes 22 by 4 to 30 %.
  const bool large_weight = (double)(N * K) > l.mid_wavesplit_max_weight, large = (double)M <= l.large_weight_max_tokens && large_weight;
  if (large_weight && !large && (double)M <= l.few_workgroups_max_tokens && base.family == TF_DMA &&
      ceil_div(M, best.bm) * ceil_div(N, best.bn) * best.splits <= ceil_div(M, base.bm) * ceil_div(N, base.bn) * base.splits)
    return TileChoice{TF_NONE, 0, 0, 1, 0.0};
  const double margin = base.family == TF_TWO_PHASE ? l.two_phase_margin : large ? l.large_weight_margin : l.margin;
  return best.us < margin * base_us ? best : TileChoice{TF_NONE, 0, 0, 1, 0.0};
}

// A second look at what was chosen (the swept tile, or `base` where that stays) where the weight is large enough to come from
// memory: 64 x 128 tiles on one CU in two read it at 33 KB a microsecond and CU, whatever their MFMAs could take, so what counts is
// how many CUs read and how often each row is fetched, which the times above know little of.  Fitted to 19 000 timings of 330
// shapes with 40 to 400 million weights, 17 to 1500 tokens: 3 to 4 % root mean square, where the times above are off by 5 to 7.
// Within 8 % it does not order two tiles.
// A weight below 80 million bytes may also lie in the 256 MB Infinity Cache (the few layers of a small model, or three in turn), where the
// times above are the better ones: a tile is taken only if it models at most `cold_cached` times as long by those too.  That is where the
// tiles measure the same with three weights in turn, 1.08 for the scaled kinds and 1.03 for the others, at 400 shapes of 40 to 100 million
// weights: with it linears take 0.966 (scaled) and 0.992 as long with three in turn, 0.905 and 0.966 with weights from memory; without it
// INT8 and epilogue scales take 1.044 with three in turn (143 tokens 7168 -> 9216 21.8 / 27.2 us in three K splits, and 30.2 / 34.1 from
// memory; 191 tokens 9216 -> 7168 26.4 / 30.4, but 39.7 / 36.1).  From 80 million on three weights leave the cache: 0.93 and 0.91.
// What it changes, 300 shapes with the layers of 64 to 66 million weights among them (profiles/tile_choice_large_weights.txt): 0.942 with three
// in turn, at most 1.11, 0.899 from memory, at most 1.05.  us from memory, before / after: block FP8 139 tokens 18432 -> 7168 52.5 / 45.9,
// 158 tokens 16640 -> 16384 104.6 / 77.7, 115 tokens 7680 -> 9600 37.0 / 30.0; per-token FP8 510 tokens 3456 -> 16512 51.9 / 44.2;
// INT8 169 tokens 7168 -> 36864 98.4 / 83.4.
// Not judged: the 256 x 256 tile where it was chosen (2556 tokens 7168 -> 7168 155.3, 128 x 192 tiles 159.0), the INT8 kernel of 128 x 256 tiles in two phases, which has no time of its own here, and up to 128 tokens a split plan that
// fills seven eighths of the chip, where two token tiles cost less than `cold_again` has it (128 tokens 18432 -> 7168: 64 x 128 tiles
// in two splits 49.8 us measured, 128 x 128 in four 44.2; modelled 48 and 39; 72 tokens 8320 -> 21120 44.8 against 46.3).
TileChoice choose_cold_tile(GemmKind kind, int64_t M, int64_t N, int64_t K, const TileChoice& base, const TileChoice& swept) {
  const TileTimes& t = tile_times(kind);
  const TileLimits& l = tile_model().limits;
  const TileChoice& c = swept.family != TF_NONE ? swept : base;
  if ((double)(N * K) < l.cold_min_weight || c.family == TF_NONE || c.family == TF_TWO_PHASE) return swept;
  if (kind == GK_INT8 && swept.family == TF_NONE && c.bm == 128 && c.bn == 256) return swept;
  if ((double)M <= l.cold_full_max_tokens && c.family == TF_DMA && c.splits > 1 &&
      (double)(ceil_div(M, c.bm) * ceil_div(N, c.bn) * c.splits) >= l.cold_full_workgroups)
    return swept;
  const auto cold = [&](int family, int i, int splits, double most) {
    return family == TF_WAVESPLIT ? cold_wavesplit_tile_us(t, i, M, N, K, most) : cold_dma_tile_us(t, i, M, N, K, splits, most);
  };
  const auto cached = [&](int family, int i, int splits) {
    return family == TF_WAVESPLIT ? wavesplit_tile_us(t, i, M, N, K) : dma_tile_us(t, i, M, N, K, splits);
  };
  int index = -1;  // of the tile to be beaten
  if (c.family == TF_DMA)
    for (int i = 0; i < 13; ++i)
      if (MID_TILES[i].bm == c.bm && MID_TILES[i].bn == c.bn) index = i;
  if (c.family == TF_WAVESPLIT)
    for (int i = 0; i < WAVESPLIT_MODELLED; ++i)
      if (WAVESPLIT_TILES[i].bm == c.bm && WAVESPLIT_TILES[i].bn == c.bn) index = i;
  if (index < 0) return swept;
  const double most = l.cold_margin * cold(c.family, index, c.splits, 1e30);  // (within that it does not order two tiles)
  const double limit = (double)(N * K) >= l.cold_only_min_weight ? 1e30 : t.cold_cached * cached(c.family, index, c.splits);
  const auto allowed_us = [&](int family, int i, int splits, double least) {
    const double u = cold(family, i, splits, least);
    return u < least && limit < 1e30 && cached(family, i, splits) > limit ? 1e30 : u;
  };
  TileChoice best = fastest_dma_tile(M, N, K, [&](int i, int splits, double least) { return allowed_us(TF_DMA, i, splits, least); }, most);
  if (wavesplit_allowed(M, N, K)) {
    const TileChoice ws = fastest_wavesplit_tile([&](int i, double least) { return allowed_us(TF_WAVESPLIT, i, 1, least); }, best.us);
    if (ws.family != TF_NONE) best = ws;
  }
  const double two_phase = M > 128 && two_phase_us(t, M, N, K) <= limit ? cold_two_phase_us(t, M, N, K) : 1e30;
  if (two_phase < best.us) best = {TF_TWO_PHASE, 256, 256, 1, two_phase};
  return best.family != TF_NONE ? best : swept;
}

// The same, or the kernel that keeps the weight in registers where the call allows it and it models 7 % faster than what would run.  Its modelled
// times are of the loop it had before its outputs became kernels of their own, and longer than it takes now: a call that is not taken may have gained by it,
// one that is taken rarely loses (114 random linears of K = 768 that take it 0.85 of the time in a graph, seven slower, by up to 7 %).
// Linears on both sides of the line, us in a graph, other / this, taken: block FP8 368 tokens 512 -> 32768 19.5 / 16.6; packed exponents 1493 tokens
// 768 -> 7296 21.2 / 17.4; per-token FP8 827 tokens 768 -> 24576 38.0 / 28.9; INT8 577 tokens 768 -> 20496 25.0 / 22.7, 975 tokens 768 -> 65584 120 / 102,
// 1100 tokens 108 / 102.  Not taken: block FP8 430 tokens 512 -> 24576 18.0 / 14.9, 458 tokens 512 -> 16384 13.3 / 11.6, 1544 tokens 512 -> 4096 13.5 / 11.8,
// 849 tokens 512 -> 6144 11.1 / 11.0, 784 tokens 512 -> 5184 10.7 / 10.9, 40 tokens 768 -> 34944 10.6 / 11.3; per-token FP8 624 tokens 640 -> 16384
// 18.3 / 14.6, 180 tokens 512 -> 24576 10.4 / 11.2; INT8 4088 tokens 768 -> 1856 17.1 / 18.7.
TileChoice choose_mid_tile(GemmKind kind, int64_t M, int64_t N, int64_t K, const TileChoice& base, bool resident_allowed) {
  double base_us;
  const TileChoice c = choose_cold_tile(kind, M, N, K, base, choose_swept_tile(kind, M, N, K, base, base_us));
  if (!resident_allowed) return c;
  const TileChoice r = best_resident(kind, M, N, K);
  return r.us < tile_model().limits.resident_margin * (c.family != TF_NONE ? c.us : base_us) ? r : c;
}

// Up to 16 tokens on a weight large enough to be loaded as a stream (streams_weight): the wave-split and the mid-M tile have such loads, the
// register wave-split kernel and the streaming kernel, whose instructions fetch parts of lines, lose by them.  Fitted to 290 linears
// (100 to 480 million weights): 3 % root mean square; what it chooses takes 1.01 of the best one's time.
// us, before / this: 18432 -> 14336 at 1 and 16 tokens block FP8 53.5 / 45.2, 64.1 / 47.9, INT8 55.7 / 44.4, 73.7 / 48.9; 8192 -> 14336 at 4 block
// 36.8 / 23.4, packed exponents 29.3 / 23.4; 7168 -> 36864 at 4 INT8 53.2 / 44.2; 7168 -> 24576 at 8 per-token FP8 40.5 / 32.2; 12672 -> 14208 at 1
// per-token FP8 40.2 / 30.1.
// One and two tokens stay on the register kernel where their K is one of its turns of 32 blocks and its quantizer saves the launch (at 1: 3584 -> 36864
// 23.3 / 24.8; at 2: 4096 -> 28672 23.5 / 24.5; one token, 24 to 32 blocks, 64 linears 1.01).  From the second turn on they do not: 118 linears of
// one token, 33 to 63 blocks, 0.92 (7552 -> 16384 24.2 / 21.9, 7168 -> 36864 48.9 / 47.0; at most 1.06, 16.5 to 20 thousand channels, which are a
// second round of the tile), longer K on fewer than 11000 channels 0.81 (0.72 to 0.90), weights of 100 to 105 million 0.84 (0.70 to 0.95).
bool streamed_decode(int64_t M, int64_t N, int64_t K) {
  const TileLimits& l = tile_model().limits;
  if (M > 16 || K % KSTEP != 0 || N % 16 != 0 || (double)(N * K) < l.streamed_min_weight) return false;
  return M > 2 || (double)ceil_div(K, KSTEP) >= l.streamed_two_tokens_min_kblocks;
}
double streamed_mid_us(int64_t M, int64_t N, int64_t K, int bn) {
  const StreamedTimes& t = tile_model().streamed;
  const int64_t wg = ceil_div(N, bn);
  const bool two = bn == 128 && wg > NUM_CUS;
  const double us = t.launch + (double)ceil_div(wg, two ? 2 * NUM_CUS : NUM_CUS) * (double)ceil_div(K, KSTEP) *
                                   (t.block + bn * t.block_channel + (double)M * t.block_token) * (two ? t.shared : 1.0);
  return norm_of(us, (double)(N * K) * 1e-6 / t.mid_stream + t.mid_stream_us, 6.0);
}
double streamed_wavesplit_us(int64_t M, int64_t N, int64_t K, int bn) {
  const StreamedTimes& t = tile_model().streamed;
  const double us = (double)ceil_div(N, (int64_t)bn * NUM_CUS) * (t.tile + (double)K * 1e-3 * (bn * t.channel + (double)M * t.token));
  return norm_of(us, (double)(N * K) * 1e-6 / t.stream + t.stream_us, t.norm);
}
// `settled`: what runs without this rule where that is one of the two tiles; it stays unless another is 8 % faster (within that the model does
// not order them: 12672 -> 9728 at 2 tokens 16 x 64 25.6, 16 x 16 27.9; 7168 -> 18432 at 16 64 x 128 29.4, 16 x 32 31.2).
// Weight rows a multiple of 4096 bytes apart have no rule of their own: the mid-M tile, whose K loops start at different blocks there, is the
// faster one there too (wave-split or register kernel / mid-M tile at 4096 -> 28672, 3 to 10 tokens: per-token FP8 28.0 / 24.0, 28.8 / 24.2,
// 27.8 / 24.6, 26.3 / 24.1, INT8 26.3 / 24.2 at 4, block FP8 26.2 / 24.6 at 4, 27.8 / 24.8 at 10; 112 such linears 0.913, at most 1.02).
TileChoice choose_streamed_tile(int64_t M, int64_t N, int64_t K, const TileChoice& settled) {
  const TileLimits& l = tile_model().limits;
  TileChoice best{TF_NONE, 0, 0, 1, 1e30};
  const auto consider = [&](int family, int bm, int bn, double us) {
    if (family == settled.family && bn == settled.bn) us *= l.cold_margin;
    if (us < best.us) best = {family, bm, bn, 1, us};
  };
  for (int i = 0; i < 3; ++i) consider(TF_WAVESPLIT, 16, WAVESPLIT_TILES[i].bn, streamed_wavesplit_us(M, N, K, WAVESPLIT_TILES[i].bn));
  for (int bn = 128; bn <= 256; bn += 64)  // (in one round: 2048 -> 67232 at 13 in 351 workgroups 34.6, the register kernel 29.6)
    if (ceil_div(N, bn) <= (bn == 128 ? 2 : 1) * NUM_CUS) consider(TF_DMA, 64, bn, streamed_mid_us(M, N, K, bn));
  return best;
}

// K not a multiple of 128 (scales in the epilogue only), us before / after where it says no more (the generic kernel, or the wave-split
// tile wherever it modelled below twice the mid-M tile, before).
// Above 16 tokens the wave-split tile, or the mid-M tile with K unsplit where it models 5 % faster: per-token FP8 149 tokens 832 -> 8832
// 12.9 / 8.9, 94 tokens 5440 -> 36352 102 / 60, 236 tokens 5216 -> 15360 54 / 38, 2000 tokens 4112 -> 2048 65 / 34; INT8 426 tokens 1504 -> 27200
// 77 / 35, 173 tokens 608 -> 18816 22.7 / 10.3, 4096 tokens 4176 -> 4096 230 / 87.  The mid-M tile only from half a chip of workgroups on: with fewer
// the generic kernel's K split wins (generic / mid-M tile: 94 workgroups 16688 -> 6016 at 65 64.7 / 79.8, 102 8016 -> 13000 at 33
// 46.6 / 50.0, 76 10480 -> 9656 at 17 40.0 / 57.2; 157 10000 -> 10016 at 200 102.5 / 58.6).  `two_phase`: FP8 where the 256 x 256 tile with a
// promotion per block runs otherwise; it stays for long K (that / mid-M tile: 4096 tokens 7184 -> 18432 596 / 679, 2048 tokens 7184 ->
// 36864 618 / 676, 4112 -> 28672 315 / 319; 4096 tokens 2064 -> 18432 258 / 229, 1040 -> 16384 152 / 120, 3000 tokens 720 -> 12288 86 / 57).  K
// below two blocks is no layer's and stays where it was.
// Up to 16 tokens the wave-split tile; from `streamed_min_weight` on what the weight's stream chooses: 14304 -> 19776 at 4 76.3 / 62.8, 8464 ->
// 22208 at 1 57.6 / 42.8, 7776 -> 18688 at 9 46.8 / 39.4.
TileChoice choose_ragged_tile(int64_t M, int64_t N, int64_t K, bool two_phase) {
  const TileTimes& t = tile_model().plain;
  const TileLimits& l = tile_model().limits;
  const TileChoice none{TF_NONE, 0, 0, 1, 0.0};
  const double weights = (double)(N * K);
  if (M <= 16 && weights >= l.streamed_min_weight) return choose_streamed_tile(M, N, K, none);
  const TileChoice ws = best_wavesplit_tile(t, M, N, K);
  const bool ws_allowed = weights <= l.ragged_max_weight && ws.us < l.ragged_max_factor * best_dma_tile(t, M, N, K).us;
  if (M > 16 && (double)ceil_div(K, KSTEP) >= l.ragged_min_kblocks) {
    TileChoice d{TF_NONE, 0, 0, 1, ws_allowed ? l.margin * ws.us : 1e30};
    if (two_phase && weights > l.ragged_max_weight && (double)ceil_div(K, KSTEP) > l.ragged_two_phase_kblocks) return none;
    for (int i = 0; i < 13; ++i) {
      const int bm = MID_TILES[i].bm, bn = MID_TILES[i].bn;
      if ((double)(ceil_div(M, bm) * ceil_div(N, bn)) < l.ragged_min_workgroups) continue;
      const double us = dma_tile_us(t, i, M, N, K, 1, d.us);
      if (us < d.us) d = {TF_DMA, bm, bn, 1, us};
    }
    if (d.family == TF_DMA) return d;
  }
  return ws_allowed ? ws : none;
}

// K of up to 16 blocks on weights of up to 20 million values, which the launches bound: the tile quantizes the tokens in its one launch and takes
// their scales as they lie.  600 linears of 1 to 16 tokens, the tile's time by what it takes over from (geometric mean, and range):
//   the register kernel: K below 8 blocks FP8 0.61 (0.40 to 0.76), INT8 0.84 (0.41 to 0.99); from 8 blocks on 0.86 (0.73 to 1.00) from five tokens
//   on, 1.01 (0.71 to 1.18) up to four; with more than five pieces of eight values a thread (20800 in all) the quantizer in every workgroup
//   takes longer than its launch (2048 -> 4096 at 16 tokens 5.8 / 8.2);
//   the streaming kernel: 0.61 (0.49 to 0.83) up to one round of its widest tile, 16384 channels; beyond, 1.19 (0.82 to 1.27; packed exponents
//   640 -> 16896 at 16 tokens 8.3 / 10.0).
bool small_decode(int64_t M, int64_t N, int64_t K, bool from_wavesplit, bool from_streaming) {
  const TileLimits& l = tile_model().limits;
  const int64_t kb = ceil_div(K, KSTEP);
  if (M > 16 || K % KSTEP != 0 || (double)(N * K) > l.decode_short_max_weight || (double)kb > l.decode_min_kblocks) return false;
  if (from_streaming) return (double)N <= l.small_max_channels;
  return from_wavesplit && ((double)kb < l.decode_short_min_kblocks || ((double)M > l.small_min_tokens && (double)(M * K) <= l.small_max_tokens_values));
}
// Up to 16 tokens, eight channels a workgroup instead of sixteen where twice the workgroups still make one round: each loads half the weight rows through
// a CU that takes 100 KB a microsecond.  us in a graph, 16 / 8: block FP8 7168 -> 576 at 1 token 4.59 / 4.50, 7168 -> 896 at 2 5.49 / 5.20; per-token FP8 7680 -> 1792 at 2
// 6.25 / 5.98; INT8 7168 -> 576 at 12 7.62 / 7.34; packed exponents 7168 -> 192 at 1 4.60 / 4.35; 45 linears 0.974, at most 1.01 (nine tokens and more, which the
// quantizer in the tile bounds).  From 24 blocks of K on, three for each wave: 96 linears of 64 to 2048 channels, graph, by blocks 4 to 16 1.006 (1.00 to 1.01),
// 17 to 22 0.996 (0.98 to 1.00), 24 0.990, 25 0.986, 28 0.985.
TileChoice half_decode_tile(int64_t M, int64_t N, int64_t K, TileChoice c) {
  const TileLimits& l = tile_model().limits;
  if (c.family == TF_WAVESPLIT && c.bm == 16 && c.bn == 16 && M <= 16 && ceil_div(N, 8) <= NUM_CUS && (double)ceil_div(K, KSTEP) >= l.half_decode_min_kblocks &&
      (double)(N * K) < l.streamed_min_weight)
    c.bn = 8;
  return c;
}
TileChoice best_decode_tile(GemmKind kind, int64_t M, int64_t N, int64_t K) {
  const TileTimes& t = tile_times(kind);
  TileChoice best{TF_NONE, 0, 0, 1, 1e30};
  for (int i = 0; i < 3; ++i) {
    static_assert(WAVESPLIT_TILES[2].bm == 16, "the 16-token tiles come first");
    const double us = wavesplit_tile_us(t, i, M, N, K, best.us);
    if (us < best.us) best = {TF_WAVESPLIT, WAVESPLIT_TILES[i].bm, WAVESPLIT_TILES[i].bn, 1, us};
  }
  return half_decode_tile(M, N, K, best);
}

// Up to 16 tokens: the wave-split tile against the kernel the constants table names.  It wins over the streaming and the register
// wave-split kernel wherever K has more than 16 blocks and the weight is not one of the largest (us, the other / the tile, one
// token and 16; FP8):
//   K = 7168: N = 576 6.8/5.1, 9.4/5.6;  2048 6.9/5.2, 8.8/6.5;  K = 14336: N = 512 9.9/6.8, 8.0/6.8;  K = 5120: N = 10240 16.0/10.2, 13.9/10.5
//   K = 18432: N = 896 12.4/7.7, 11.6/9.4;  7168 23.3/23.1, 28.1/25.0;  K = 4096: N = 6144 7.5/6.3, 9.7/6.2;  28672 22.9/24.7, 26.1/25.5
// because its operands come in whole 128-byte lines: 16 rows x 64 bytes per instruction, which is what the MFMA's layout asks
// for when loaded straight into registers, pass through a CU's cache at 16 bytes a cycle, whole lines at 61.
// With fewer K blocks both are bound by the launch (K = 2048 -> N = 2048 4.3 / 4.4) except where there are many channels
// (K = 1024 -> N = 12288 5.8/4.8, 8.0/4.9; but 512 -> 32768 5.9/6.8, 1536 -> 24576 9.3/9.6).
// It does not take over from
//   * the mid-M kernel, which the table names where one round of unsplit tiles fills the chip (K = 2304 -> N = 36864 at 16 tokens
//     19.3/22.9, 5120 -> 50688 51.3/57.3, INT8 1024 -> 17408 at 12 tokens 7.1/9.0; over 91 shapes 6 % faster), also where the rows of the weight
//     lie a multiple of 4096 bytes apart: its K loops start at different blocks there (4096 -> 30464 23.5/25.7, per-token FP8 23.9/25.1;
//     linears of 12 to 16 tokens, 4096 -> 18432 .. 32768, 95 of them: 0.90, at most 1.02);
//   * the register wave-split kernel where K fills its one turn of 32 blocks and the channels are more than one round of the widest tile,
//     up to 10 tokens: 4096 -> 20736 at 1 and 8 19.0/24.4, 21.3/24.4; 3840 -> 24576 at 1 20.0/23.0 (4096 -> 16384 at 1, 8 14.8/16.3,
//     16.3/16.3; 3584 -> 27392 at 6 23.6/21.8).
// The weight limits were drawn at the shapes named beside them.  Measured around them since (K = 2304 .. 18432, 85 to 260 million weights,
// 1 .. 16 tokens): also beyond them the tile is up to 25 % faster than the streaming and the two-turn register kernel, and slower than
// the one-turn one; but a linear that leaves those loses their fused quantizers, so the limits stay where the linears were measured.
TileChoice choose_limited_decode_tile(GemmKind kind, int64_t M, int64_t N, int64_t K, bool from_mid, bool from_wavesplit, bool from_streaming) {
  const TileLimits& l = tile_model().limits;
  const int64_t kb = ceil_div(K, KSTEP);
  const double weight = (double)(N * K);
  // (the largest weights: the register kernel's single-tile stream is as fast for few tokens, unless it pads K to whole turns of 32 blocks:
  // K = 5152 -> N = 31936 INT8 at 5 tokens 50.3 us, 39.3 with the tile)
  const bool padded = kb <= 64 && (kb + 31) / 32 * 32 * 4 > kb * 5;
  if (from_mid) return TileChoice{TF_NONE, 0, 0, 1, 0.0};
  const bool one_turn = (double)kb >= l.decode_one_turn_min_kblocks && (double)kb <= l.decode_one_turn_kblocks;
  if (from_wavesplit && one_turn && (double)M <= l.decode_one_turn_max_tokens && (double)N > l.decode_one_turn_max_channels)
    return TileChoice{TF_NONE, 0, 0, 1, 0.0};
  const bool few = (double)M <= (kind == GK_F32 ? l.decode_few_tokens_f32 : l.decode_few_tokens) && (double)kb <= l.decode_long_kblocks;
  const double most = padded ? l.decode_padded_max_weight : few ? l.decode_few_tokens_max_weight : l.decode_max_weight;
  const bool small = small_decode(M, N, K, from_wavesplit, from_streaming);
  const bool take = small || ((double)kb > l.decode_min_kblocks ? weight <= most
                                                      : (double)kb >= l.decode_short_min_kblocks && (double)N >= l.decode_short_min_channels &&
                                                            weight <= l.decode_short_max_weight && (double)M > l.decode_short_min_tokens);
  if (!take) return TileChoice{TF_NONE, 0, 0, 1, 0.0};
  return best_decode_tile(kind, M, N, K);
}

// `base`: what the constants table names.
TileChoice choose_decode_tile(GemmKind kind, int64_t M, int64_t N, int64_t K, const TileChoice& base, bool from_wavesplit, bool from_streaming) {
  const TileChoice c = choose_limited_decode_tile(kind, M, N, K, base.family == TF_DMA, from_wavesplit, from_streaming);
  // (a bare GEMM with fp32 scales keeps its kernel: the mid-M tile may need a launch that lays the token scales out again.  The one-call
  // linear of that kind lays them out as it likes: choose_linear.)
  if (kind == GK_F32 || !streamed_decode(M, N, K)) return c;
  return choose_streamed_tile(M, N, K, c.family != TF_NONE ? c : base);
}

}  // namespace
}  // namespace mi355
