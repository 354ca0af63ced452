// Mid-M FP8 GEMM for gfx950: the tile of gemm_dma_tile.h with fp32 block scales, packed UE8M0 scales applied by the MFMA, or
// one scale per token and channel applied in the epilogue; its grouped form; the one-call linear at decode sizes, whose
// producer waves quantize the tokens; and the choice of tile and K split.
//
// For 16 < M <= 1024 a linear layer is between weight streaming and MFMA-bound; prefill shapes with few output channels
// (M = 4096, N = 576 or 1536) do not give 256 x 256 tiles enough workgroups.  Both take this kernel.  The tile is short in the
// token dimension and wide in channels (256; 192 and 128 where those fill the chip better: 36864 channels are 144 tiles of 256
// but 192 of 192, 1536 channels x 4096 tokens are exactly 256 tiles of 128 x 192).  Optional split along K (partials to the
// workspace, ordered reduce afterwards).
// Requires K % 128 == 0, 16-byte aligned rows, row offsets below 4 GiB, and token scales laid out M-major with a pitch that is
// a multiple of four floats (fp8_scales_conform; the dispatcher re-lays other layouts out into the workspace first).
#include "gemm_dma_tile.h"

namespace mi355 {
namespace {

constexpr int T_BN = 256;  // widest channel tile

template <int BM, int BN>
struct Dma3State {
  static constexpr int LOADS = (BM + BN) / 64;  // tile loads per wave and stage (a wave fills 8 rows per load)
  const uint8_t* b_base;
  uint32_t goff[LOADS];   // lane's byte offset from the matrix base (rows clamped); the first BM / 64 (token rows) are not used
  // Weight-block scale rows.  A wave's channels are BN / 4 consecutive ones inside one 128-channel block, except for
  // BN = 192, where 48 consecutive channels could straddle two blocks: there the wave's tile i is channels
  // 64 i + 16 wave .. + 15 of the tile, so that tile i of every wave lies in the block of channel n0 + 64 i.
  static constexpr bool INTERLEAVED = BN == 192;
  static constexpr int SB = INTERLEAVED ? BN / 64 : 1;
  static constexpr int W_STRIDE = INTERLEAVED ? 64 * 128 : 16 * 128;  // bytes between a wave's consecutive channel tiles in a stage
  cfloat_ptr sb_ptr[SB];  // &sb[nb, 0] of the wave's (tile's) 128-channel block
  int64_t sb_sk;
  int wave, kb_last;
  uint32_t tok_off[2], ch_off[2], sc_off;
};

// ---- pieces of the producer-wave kernel (dma3_tile_q below), whose K block reads its fragments and multiplies them in turn.
// Load number i (a tile-row load) of K block kb, written as instructions.
// The statements write m0; it cannot be listed as a clobber (the compiler reserves the register and rejects the entry), and
// no compiler-managed use of m0 lies between them and the next statement that sets it.
template <int BM, int BN, bool STREAM>
__device__ __forceinline__ void issue_one(const Dma3State<BM, BN>& s, int i, uint8_t* stage, int kb) {
  kb = min(kb, s.kb_last);
  const uint8_t* base = s.b_base + (uint64_t)kb * KSTEP;  // wave-uniform
  asm volatile("" : "+s"(base));
  const uint32_t lds_addr = (uint32_t)(uintptr_t)(lptr_t)(stage + (i * 64 + s.wave * 8) * KSTEP);
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(s.goff[i]), "s"(base), "s"(lds_addr) : "memory");
  else
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(s.goff[i]), "s"(base), "s"(lds_addr) : "memory");
}

// One K block out of `cur`; the weight-row loads of block kb_next go out in between, into `nxt` (a producer wave writes the
// token rows).
template <int BM, int BN, bool STREAM>
__device__ __forceinline__ void k_block(const Dma3State<BM, BN>& s, const uint8_t* cur, const float* sc_cur,
                                        const float (&sbv)[Dma3State<BM, BN>::SB], float (&acc)[BN / 64][BM / 32][4], uint8_t* nxt,
                                        int kb_next) {
  constexpr int MT = BM / 32, T_NT = BN / 64, LOADS = Dma3State<BM, BN>::LOADS;  // a wave owns BN / 4 channels = T_NT tiles of 16
  constexpr int SB = Dma3State<BM, BN>::SB, W_STRIDE = Dma3State<BM, BN>::W_STRIDE;
  static_assert(LOADS <= MT * T_NT, "one load per step");
  Frag w[T_NT], tokb[2];
  float scb[2][SB];
  const lds_cptr ch0 = (lds_cptr)cur + s.ch_off[0], ch1 = (lds_cptr)cur + s.ch_off[1];
  const lds_cptr tk0 = (lds_cptr)cur + s.tok_off[0], tk1 = (lds_cptr)cur + s.tok_off[1];
  w[0].lo = lds16(ch0, 0);
  w[0].hi = lds16(ch1, 0);
  tokb[0].lo = lds16(tk0, 0);
  tokb[0].hi = lds16(tk1, 0);
  const float* scp = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(sc_cur) + s.sc_off);
#pragma unroll
  for (int b = 0; b < SB; ++b) scb[0][b] = scp[0] * sbv[b];
  __builtin_amdgcn_sched_barrier(0);

  v4f part[2];
#pragma unroll
  for (int t = 0; t < MT * T_NT; ++t) {
    const int j = t / T_NT, i = t % T_NT;
    part[t & 1] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(as_v8i(w[i]), as_v8i(tokb[j & 1]), v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0,
                                                                   0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // the MFMA goes first; the rest of the step runs in its shadow
    if (t > 0) {
      const int pj = (t - 1) / T_NT, pi = (t - 1) % T_NT;
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[pi][pj][v] = fmaf(part[(t - 1) & 1][v], scb[pj & 1][SB > 1 ? pi : 0], acc[pi][pj][v]);
    }
    if (t + 1 < T_NT) {  // remaining weight fragments, one per step
      w[t + 1].lo = lds16(ch0, (t + 1) * W_STRIDE);
      w[t + 1].hi = lds16(ch1, (t + 1) * W_STRIDE);
    }
    if (i == 0 && j + 1 < MT) {  // next token tile
      tokb[(j + 1) & 1].lo = lds16(tk0, (j + 1) * 2048);
      tokb[(j + 1) & 1].hi = lds16(tk1, (j + 1) * 2048);
    }
    if (i == 1 && j + 1 < MT) {
#pragma unroll
      for (int b = 0; b < SB; ++b) scb[(j + 1) & 1][b] = scp[(j + 1) * 16] * sbv[b];
    }
    if (t >= BM / 64 && t < LOADS) issue_one<BM, BN, STREAM>(s, t, nxt, kb_next);
    __builtin_amdgcn_sched_barrier(0);
  }
  constexpr int t = MT * T_NT - 1;
  constexpr int pj = t / T_NT, pi = t % T_NT;
#pragma unroll
  for (int v = 0; v < 4; ++v) acc[pi][pj][v] = fmaf(part[t & 1][v], scb[pj & 1][SB > 1 ? pi : 0], acc[pi][pj][v]);
}

// Everything but the YOUNGER youngest loads has landed; then the workgroup barrier.  Instructions, see the file comment.
template <int YOUNGER>
__device__ __forceinline__ void wait_and_barrier() {
  static_assert(YOUNGER >= 4 && YOUNGER <= 28, "(stages - 2) x (LOADS + 1), LOADS + 1 = (BM + BN) / 64 + 1");
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
}

// Epilogue of its compute waves: the lane holds channels n .. n+3 of token m for each of its MFMA tiles (at most 16 tokens are
// stored: not worth a pass through LDS).
template <int BM, int BN>
__device__ __forceinline__ void store_tile(const GemmParams& p, float (&acc)[BN / 64][BM / 32][4], int m0, int n0, int wave_m, int wave_n,
                                           int l16, int q) {
  constexpr int WM = BM / 2, MT = WM / 16, T_WN = BN / 4, T_NT = T_WN / 16;
  constexpr bool INTERLEAVED = Dma3State<BM, BN>::INTERLEAVED;
  const bool vec_ok = ((p.ldo & 3) == 0) && ((reinterpret_cast<uintptr_t>(p.out) & 15) == 0);
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int m = m0 + wave_m * WM + j * 16 + l16;
    if (m >= p.M) continue;
#pragma unroll
    for (int i = 0; i < T_NT; ++i) {
      const int n = n0 + (INTERLEAVED ? i * 64 + wave_n * 16 : wave_n * T_WN + i * 16) + 4 * q;
      if (n >= p.N) continue;
      fp8_channel_epilogue(p, n, acc[i][j]);
      store_out4(p.out, p.out_dtype, (int64_t)m * p.ldo + n, acc[i][j], min(4, p.N - n), vec_ok);
    }
  }
}

// ---- The 64-token tile for the one-call linear at decode sizes (M <= 16, K unsplit): the tokens arrive unquantized
// (p.x16, bf16 or fp16) and four more waves, the PRODUCERS, quantize the 16 x 128 values of a K block into the stage's token rows
// and scale slots - the arithmetic of the group quantizer's reference path (quantize_group_lane), so the result equals
// quantizer launch + GEMM bit for bit - while waves 0..7 load the weight rows and multiply as above.  A producer requests
// the raw tokens four blocks ahead of the one it quantizes (one 16-byte load per lane and block, its own vmcnt), writes S - 1 blocks ahead of
// the one being multiplied, and meets the others at every block's barrier.  Token rows 16..63 of a stage are never written:
// what they hold only reaches accumulators of rows that are not stored.
constexpr int T_PW = 4;  // producer waves of the fused quantizer
template <int BN, int S, bool STREAM>
__device__ __forceinline__ void dma3_tile_q(const GemmParams& p, int n0) {
  constexpr int BM = 64;
  static_assert(S >= 3 && S * ((BM + BN) * KSTEP + BM * 4) <= 160 * 1024, "the stages must fit the CU's LDS");
  constexpr int LOADS = Dma3State<BM, BN>::LOADS, LOADS_W = LOADS - BM / 64;  // weight-row loads per wave and block
  constexpr bool INTERLEAVED = Dma3State<BM, BN>::INTERLEAVED;
  constexpr int SB = Dma3State<BM, BN>::SB, WM = BM / 2, MT = WM / 16, T_WN = BN / 4, T_NT = T_WN / 16;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nkb = p.kb_total, kb_last = p.kb_total - 1;

  __shared__ __attribute__((aligned(1024))) uint8_t t_stage[S][(BM + BN) * KSTEP];
  __shared__ __attribute__((aligned(256))) float t_scale[S][BM];

  if (wave >= 8) {
    // ================= producer wave pw: tokens 4 pw .. 4 pw + 3 =================
    // (one wave quantizing all sixteen tokens of a block takes ~1.3 us of dependent arithmetic per block, more than the block's
    // multiplication: 78 against 50 us on K=7168 -> N=36864; four waves take a quarter each)
    const int pw = wave - 8;
    const int gl = lane & 15, r4 = lane >> 4;  // 16 lanes per (token, block) group; four tokens per wave
    const int m = pw * 4 + r4;                 // the stage row this lane's group goes to; rows past M repeat the last token
    const bool active = pw * 4 < p.M;          // a wave whose tokens all lie past M only keeps the barriers
    const uint16_t* xrow = reinterpret_cast<const uint16_t*>(p.x16) + (int64_t)min(m, p.M - 1) * p.ldx + gl * 8;
    auto request = [&](int kb, u32x4& raw) {
      const uint16_t* src = xrow + (int64_t)min(kb, kb_last) * KSTEP;
      asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(raw) : "v"(src) : "memory");
    };
    auto produce = [&](int stage, const u32x4& raw) {
      float sc;
      const u32x2 codes = quantize_group_lane(raw, p.x_dtype, p.x_by_reciprocal != 0, sc);
      *reinterpret_cast<u32x2*>(&t_stage[stage][m * KSTEP + (((gl >> 1) ^ (m & 7)) << 4) + (gl & 1) * 8]) = codes;
      if (gl == 0) t_scale[stage][m] = sc;
    };
    // A ring of R registers keeps the raw tokens of the next R blocks in flight: one is quantized into its stage, then
    // requested again for the block R further on (a register that a load is still writing cannot be copied, so the loop is
    // unrolled over the ring).  Step b produces block b into stage b % S; from step S - 2 on (blocks 0 .. S-2 are in LDS) every
    // step ends at a barrier: the first is the one the other waves pass before block 0, the j-th after it ends their block j - 1,
    // so block b is written after the barrier that ends block b - S, the last reader of its stage.
    constexpr int R = 4;
    static_assert(R == 4, "the wait below is written for a ring of four loads");
    u32x4 ring[R];
    if (active) {
#pragma unroll
      for (int u = 0; u < R; ++u) request(u, ring[u]);
    }
    const int steps = nkb + S - 2;
    int st = 0;
    for (int b = 0; b < steps; b += R) {
#pragma unroll
      for (int u = 0; u < R; ++u) {
        if (b + u < steps) {
          if (active) {
            asm volatile("s_waitcnt vmcnt(3)" : "+v"(ring[u])::"memory");  // the oldest of the R loads in flight
            produce(st, ring[u]);
            st = st + 1 == S ? 0 : st + 1;
            request(b + u + R, ring[u]);
          }
          if (b + u >= S - 2) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
      }
    }
    if (nkb % S == 0) asm volatile("s_barrier" ::: "memory");  // the other waves' barrier after the last block of a whole trip
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }

  // ================= waves 0..7: weight loads and arithmetic =================
  const int wave_m = wave >> 2, wave_n = wave & 3;
  const int l16 = lane & 15, q = lane >> 4;
  Dma3State<BM, BN> s;
  s.wave = wave;
  s.kb_last = kb_last;
  s.b_base = p.b;
  {
    const int lrow = lane >> 3;
    const int chunk_byte = ((lane & 7) ^ lrow) * 16;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int row = i * 64 + wave * 8 + lrow;
      s.goff[i] = row < BM ? 0u : (uint32_t)((int64_t)min(n0 + row - BM, p.N - 1) * p.ldb + chunk_byte);
    }
    const int trow = wave_m * WM + l16, crow = BM + wave_n * (INTERLEAVED ? 16 : T_WN) + l16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s.tok_off[h] = trow * KSTEP + (((q + 4 * h) ^ (trow & 7)) << 4);
      s.ch_off[h] = crow * KSTEP + (((q + 4 * h) ^ (crow & 7)) << 4);
    }
    s.sc_off = (wave_m * WM + l16) * 4;
  }
#pragma unroll
  for (int b = 0; b < SB; ++b) {
    const int first = INTERLEAVED ? n0 + 64 * b : n0 + wave_n * T_WN;
    s.sb_ptr[b] = (cfloat_ptr)(p.sb + (int64_t)__builtin_amdgcn_readfirstlane(min(first, p.N - 1) / 128) * p.sb_sn);
  }
  s.sb_sk = p.sb_sk;
  constexpr int YOUNGER = (S - 2) * LOADS_W;

  float acc[T_NT][MT][4];
#pragma unroll
  for (int i = 0; i < T_NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;

#pragma unroll
  for (int b = 0; b < S - 1; ++b)
#pragma unroll
    for (int i = BM / 64; i < LOADS; ++i) issue_one<BM, BN, STREAM>(s, i, t_stage[b], b);
  wait_and_barrier<YOUNGER>();  // the weight rows of block 0 have landed; the producer has written blocks 0 .. S-2

  auto sb_of = [&](int kb, float (&v)[SB]) {
#pragma unroll
    for (int b = 0; b < SB; ++b) v[b] = s.sb_ptr[b][(int64_t)kb * s.sb_sk];
  };
  int k = 0;
  for (; k + S - 1 < nkb; k += S) {
    float sbv[S][SB];
#pragma unroll
    for (int u = 0; u < S; ++u) sb_of(k + u, sbv[u]);
#pragma unroll
    for (int u = 0; u < S; ++u) {
      k_block<BM, BN, STREAM>(s, t_stage[u], t_scale[u], sbv[u], acc, t_stage[(u + S - 1) % S], k + u + S - 1);
      wait_and_barrier<YOUNGER>();  // unconditional (a condition here makes the compiler sink arithmetic across blocks): when K
                                    // is a whole number of trips this is one barrier past the last block, which the producers match
    }
  }
#pragma unroll
  for (int u = 0; u < S - 1; ++u) {
    if (k + u < nkb) {
      float sbl[SB];
      sb_of(k + u, sbl);
      k_block<BM, BN, STREAM>(s, t_stage[u], t_scale[u], sbl, acc, t_stage[(u + S - 1) % S], k + u + S - 1);
      if (k + u + 1 < nkb) wait_and_barrier<YOUNGER>();
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // stray refetches must not outlive the workgroup's LDS
  store_tile<BM, BN>(p, acc, 0, n0, wave_m, wave_n, l16, q);
}

template <int BN, int S, bool STREAM>
__global__ __launch_bounds__(T_THREADS + 64 * T_PW) void fp8_gemm_dma3_q_kernel(const GemmParams p) {
  const TileCoord tc = tile_of_block(blockIdx.x, gridDim.x, 1, p.tiles_n);
  dma3_tile_q<BN, S, STREAM>(p, tc.tile_n * BN);
}

// Grouped problems (see GroupedParams): the workgroup's token tile comes from the table the plan kernel wrote, the
// operand bases move to that tile's expert, and the ordinary tile runs.
template <int BM, int BN, int S, bool STREAM>
__global__ __launch_bounds__(T_THREADS) __attribute__((amdgpu_waves_per_eu(BM + BN == 192 && S == 3 ? 4 : 2))) void fp8_grouped_dma_kernel(const GroupedParams gp) {
  GemmParams p;
  int m0, tile_n;
  if (!grouped_tile_of_block(gp, p, m0, tile_n)) return;  // the whole workgroup leaves before any barrier
  dma_tile<AR_F32, BM, BN, false, S, STREAM, false>(p, m0, tile_n * BN, 0);
}

}  // namespace

// Tile shape (64 or 128 tokens x 256 or 128 channels) and split count for this kernel.  One workgroup per CU fits (the
// LDS stages are sized for the widest tile).  Narrow channel tiles do half the multiplications of a block in 0.6 of the
// time, but they double the workgroups without a K split, i.e. without fp32 partial sums: they win for few channels and
// long K (K=18432 -> N=7168 at M=128: 52.7 -> 46.7 us; K=7168 -> N=4096 at M=512: 34.4 -> 24.5 us; N=576 at M=4096:
// 35.7 -> 31.0 us) and lose where 256-channel tiles already give a round's worth of workgroups.
//
// The choice minimises a time model fitted to measurements on this part (24 shapes, M = 32 .. 4096, every tile height
// and split count; it names the measured best or a choice within 5 % of it for 22 of them, within 12 % for the others):
//   * a workgroup spends per K block the largest of
//       - the tile's own time when operands come from L2: 0.88 us for 128 token rows, 0.58 us for 64 (0.52 / 0.40 with
//         128 channels, 0.68 / 0.50 with 192; x 1.2 in a round that keeps more than 200 CUs busy; the INT8 kernel: 1.14 / 0.71 / 0.64 / 0.44);
//       - a latency floor when the weight comes from HBM (two blocks in flight per CU): 1.2 us / 1.0 us (1.0 / 0.75 with 192 channels, 0.7 / 0.51 with
//         128 channels; INT8: 0.96 / 0.68 / 0.59 / 0.54), times 1.2 for weight rows longer than 8 KB;
//       - its share of the HBM stream: (concurrent workgroups) x (HBM bytes per workgroup and block) / 5.5 TB/s, where
//         weight rows are shared in L2 by up to 8 token tiles and token rows by up to 8 channel tiles;
//   * a workgroup runs kb_per + 2 blocks (pipeline fill), and rounds of up to 256 workgroups follow each other;
//   * a split adds the fp32 partial tiles written and read back (8 * splits * M * N bytes at 5.5 TB/s) and
//     8 + 0.25 * splits us for the second launch and its tail.
// So 144 workgroups streaming a weight unsplit beat 432 that split K in three (measured at M = 32 and 64 on K = 7168 ->
// N = 36864: 58 against 65 us): with all CUs busy the HBM stream, not the number of workgroups, is the limit, and the
// partial sums only add traffic.
//
// `efficiency` is the best value over all choices of an older byte-model score, kept because the dispatcher's threshold
// for preferring another kernel at M < 256 was set with it:
//   balance * useful_bytes / (useful_bytes + partial_bytes) * kb_per / (kb_per + 2) * (0.65 for 64-row tiles at M > 128)
namespace {
double dma3_model_us(int64_t M, int64_t N, int64_t kb_total, int bm, int bn, int sp, bool is_int8) {
  const RouteConstants& rc = route_constants();
  const double HBM_BYTES_PER_US = rc.dma3_hbm_bytes_per_us;
  const int64_t per = (kb_total + sp - 1) / sp;
  const int64_t tm = (M + bm - 1) / bm, tn = (N + bn - 1) / bn;
  // the tile's own time per K block and the latency floor, in the order 128x256, 64x256, 128x128, 64x128, 128x192, 64x192
  // (the INT8 kernel of the same structure has its own); the numbers and where they come from: route_constants.h
  const int shape = (bn == 256 ? 0 : bn == 128 ? 2 : 4) + (bm == 128 ? 0 : 1);  // ..., 128x192, 64x192 (FP8 only)
  const double t_tile = rc.dma3_tile_us[is_int8][shape];
  const double hbm_per_block = (double)(bn * KSTEP) / (double)std::min<int64_t>(tm, 8) + (double)(bm * KSTEP) / (double)std::min<int64_t>(tn, 8);
  // latency floor while the weight streams from HBM: with 256 or 192 channels per tile when at most two token tiles share
  // it, with 128 when nobody does (rows more than 8 KB apart cost more)
  const bool streams = hbm_per_block >= (bn == 192 ? 12288.0 : 16384.0);
  const double t_latency = streams ? rc.dma3_latency_us[is_int8][shape] * (kb_total > 64 ? rc.dma3_long_row_factor : 1.0) : 0.0;
  double t = 0.0;
  for (int64_t left = tm * tn * sp; left > 0;) {
    const int64_t c = std::min<int64_t>(left, 256);
    left -= c;
    // with (nearly) every CU multiplying, the clock drops
    const double t_own = t_tile * (c > 200 ? rc.dma3_busy_chip_factor : 1.0);
    t += (double)(per + 2) * std::max(std::max(t_own, t_latency), (double)c * hbm_per_block / HBM_BYTES_PER_US);
  }
  if (sp > 1) t += 8.0 * sp * (double)M * (double)N / HBM_BYTES_PER_US + rc.dma3_split_fixed_us + rc.dma3_split_per_split_us * sp;
  return t;
}
}  // namespace

int dma3_stages(int bm, int bn, int64_t workgroups) { return stages_of(bm, bn, workgroups <= NUM_CUS); }

Dma3Plan dma3_plan(int64_t M, int64_t N, int64_t K, bool is_int8) {
  Dma3Plan pl;
  const int64_t kb_total = (K + KSTEP - 1) / KSTEP;
  const double useful = (double)N * K + (double)M * K + 2.0 * M * N;
  const int max_split = (N % 4 == 0) ? 16 : 1;  // the reduce kernel works on aligned quads of one row
  double best_time = 1e30;
  pl.bm = 128, pl.bn = T_BN, pl.splits = 1, pl.efficiency = 0.0;
  for (int bn = T_BN; bn >= 128; bn -= 64) {
    if (bn == 192 && is_int8) continue;  // the INT8 kernel's 32-channel MFMA tiles do not divide 192 / 4
    for (int bm = 64; bm <= 128; bm += 64) {
      if (M <= 64 && bm == 128) break;                 // a second half tile of padding rows buys nothing
      const double tile_factor = (bm == 64 && M > 128) ? route_constants().dma3_small_tile_factor : 1.0;
      const int64_t tiles = ((M + bm - 1) / bm) * ((N + T_BN - 1) / T_BN);
      for (int sp = 1; sp <= max_split; ++sp) {
        const int64_t per = (kb_total + sp - 1) / sp;
        if (sp > 1 && per < 4) break;
        if ((kb_total + per - 1) / per != sp) continue;  // some split would get no work
        const double t = dma3_model_us(M, N, kb_total, bm, bn, sp, is_int8);
        if (t < best_time) best_time = t, pl.splits = sp, pl.bm = bm, pl.bn = bn;
        if (bn != T_BN) continue;  // the byte-model score below is defined on 256-channel tiles
        const int64_t wgs = tiles * sp;
        const int64_t rounds = (wgs + 255) / 256;
        const double balance = (double)wgs / (double)(rounds * 256);
        const double partial = sp > 1 ? 8.0 * sp * M * N : 0.0;
        pl.efficiency = std::max(pl.efficiency, balance * useful / (useful + partial) * (double)per / (double)(per + 2) * tile_factor);
      }
    }
  }
  pl.kb_per_split = (int)((kb_total + pl.splits - 1) / pl.splits);
  pl.time_us = best_time;
  return pl;
}

int launch_fp8_grouped_dma3(GroupedParams& gp, int bm, int bn, bool few, bool streamed, hipStream_t stream, const char* what) {
  gp.g.tiles_n = (gp.g.N + bn - 1) / bn;
  gp.g.splits = 1, gp.g.kb_per_split = gp.g.kb_total;
  const dim3 grid((unsigned)(gp.max_tiles_m * gp.g.tiles_n));
  const dim3 block(T_THREADS);
  const auto launch = [&](auto streamed) {
    constexpr bool STREAM = decltype(streamed)::value;
    if (bm == 64 && bn == 128 && few) launch_kernel((fp8_grouped_dma_kernel<64, 128, stages_of(64, 128, true), STREAM>), grid, block, 0, stream, gp);
    else if (bm == 64 && bn == 128) launch_kernel((fp8_grouped_dma_kernel<64, 128, stages_of(64, 128, false), STREAM>), grid, block, 0, stream, gp);
    else if (bn == 128) launch_kernel((fp8_grouped_dma_kernel<128, 128, stages_of(128, 128, true), STREAM>), grid, block, 0, stream, gp);
    else if (bm == 64) launch_kernel((fp8_grouped_dma_kernel<64, 256, stages_of(64, 256, true), STREAM>), grid, block, 0, stream, gp);
    else launch_kernel((fp8_grouped_dma_kernel<128, 256, stages_of(128, 256, true), STREAM>), grid, block, 0, stream, gp);
  };
  if (streamed) launch(std::true_type{});
  else launch(std::false_type{});
  return check_launch(what);
}

int launch_fp8_dma3(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_dma_tile_of<AR_F32>(p, bm, bn, stream, what);
}

// One-call linear at decode sizes: p.x16 / p.ldx / p.x_dtype describe the unquantized tokens (M <= 16, 16-byte aligned rows),
// K unsplit, one 64-token tile per workgroup; p.a and p.sa are not read.
int launch_fp8_dma3_quant(GemmParams& p, int bn, hipStream_t stream, const char* what) {
  if (p.M > 16 || p.x16 == nullptr || p.splits != 1) {
    set_error("%s: the fused quantizer of the mid-M kernel takes up to 16 unquantized tokens and an unsplit K", what);
    return MI355_ERR_UNSUPPORTED;
  }
  p.tiles_m = 1;
  p.tiles_n = (p.N + bn - 1) / bn;
  const dim3 grid((unsigned)p.tiles_n), block(T_THREADS + 64 * T_PW);
  const auto launch = [&](auto streamed) {
    constexpr bool STREAM = decltype(streamed)::value;
    if (bn == 128) launch_kernel((fp8_gemm_dma3_q_kernel<128, 6, STREAM>), grid, block, 0, stream, p);
    else if (bn == 192) launch_kernel((fp8_gemm_dma3_q_kernel<192, 4, STREAM>), grid, block, 0, stream, p);
    else launch_kernel((fp8_gemm_dma3_q_kernel<256, 3, STREAM>), grid, block, 0, stream, p);
  };
  if (streams_weight(p)) launch(std::true_type{});
  else launch(std::false_type{});
  return check_launch(what);
}

}  // namespace mi355
