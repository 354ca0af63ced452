// The mid-M tile of the FP8 and INT8 GEMMs for gfx950: 64 .. 256 tokens x 256, 192 or 128 channels, 8 waves (two per
// SIMD), S LDS stages filled by direct-to-LDS loads, operand fragments read one K block AHEAD of their multiplication.
//
// What bounds a short tile is the chain of one K block: after the block's barrier every wave reads its operand fragments
// from LDS (96-128 KB over the workgroup, ~450 cycles at the LDS's rate) and only then multiplies them (256-512 cycles of
// matrix pipe per SIMD); with eight waves in lockstep the two never overlap.  Here a wave holds two sets of fragments: while
// it multiplies block k out of one, it reads block k + 1 from LDS into the other, so the LDS and the matrix pipe work at the
// same time inside every wave and nothing but the barrier itself separates two blocks' multiplications.  The stage that
// held block k is free as soon as its fragments are in registers, so S stages keep S - 1 blocks in flight from memory as
// before.  Registers: 64 accumulators + 2 x 64 fragments for 128 x 256 (INT8 and FP8 alike), two waves per SIMD.
//
// Instructions written by hand, because the compiler's own waits cover every load it knows about:
//   * per block every wave issues exactly LOADS loads (tile rows plus, where the K loop applies scales, the token scales),
//     so "block k + 1 has landed" is the constant s_waitcnt vmcnt((S - 2) * LOADS) until the last S blocks, which issue
//     nothing and count down;
//   * s_waitcnt lgkmcnt(0) in front of the barrier: the fragments of block k have left its stage;
//   * nothing else in the loop counts in vmcnt (weight-block scales come by scalar loads).
// Requires 16-byte aligned rows and row offsets below 4 GiB; AR_F32 / AR_UE8M0 also K % 128 == 0 and token scales laid out M-major
// with a pitch that is a multiple of four words; AR_UNIT / AR_INT8 K % 128 == 0, or K % 16 == 0 in a kernel of its own (RAGGED, K not
// split): chunks past a row's end repeat its last one, and the last block's token fragments are cleared there before they are
// multiplied, so a weight row meets nothing but its own values.  One subtraction a load; what it costs is lines: rows no multiple of
// 128 bytes apart share them between K blocks (per-token FP8 94 tokens 5440 -> 36352 60, 5504 -> 36352 51 us; 102 on the generic kernel).
#pragma once

#include <utility>

#include "gemm_common.h"

namespace mi355 {
namespace {

// What the K loop does with a product block.
enum Arith {
  AR_F32,    // FP8, fp32 scales: acc += product * (token scale * weight-block scale)
  AR_UE8M0,  // FP8, packed exponents on both operands: the MFMA applies them and accumulates in place
  AR_UNIT,   // FP8, no scales in the loop: accumulates in place; one scale per token and channel in the epilogue
  AR_INT8,   // INT8: accumulates in place (int32); scales and bias in the epilogue
};

constexpr int T_THREADS = 512;

typedef __attribute__((address_space(3))) void* lptr_t;
typedef const __attribute__((address_space(3))) uint8_t* lds_cptr;
typedef const __attribute__((address_space(4))) float* cfloat_ptr;

struct Frag {
  u32x4 lo, hi;
};
__device__ __forceinline__ v8i as_v8i(const Frag& f) {
  return v8i{(int)f.lo.x, (int)f.lo.y, (int)f.lo.z, (int)f.lo.w, (int)f.hi.x, (int)f.hi.y, (int)f.hi.z, (int)f.hi.w};
}
__device__ __forceinline__ v4i as_v4i(const u32x4& x) { return v4i{(int)x.x, (int)x.y, (int)x.z, (int)x.w}; }
__device__ __forceinline__ u32x4 lds16(lds_cptr p, int imm) {
  return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(p + imm);
}
__device__ __forceinline__ float lds_f32(lds_cptr p, int imm) {
  return *reinterpret_cast<const __attribute__((address_space(3))) float*>(p + imm);
}

template <Arith AR, int BM, int BN>
struct TileShape {
  static_assert(BM % 32 == 0 && (BN == 128 || BN == 192 || BN == 256), "tile");
  static constexpr bool SCALED = AR == AR_F32 || AR == AR_UE8M0;
  // eight waves: two rows of four, or four rows of two where the tile is taller than wide (fewer fragments per product)
  static constexpr int WAVES_M = BM >= 192 && BM % 64 == 0 && BN == 128 ? 4 : 2, WAVES_N = 8 / WAVES_M;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int MT = WM / 16, NT = WN / 16, STEPS = MT * NT;   // 16 x 16 tiles of a wave
  static_assert(WM % 16 == 0 && WN % 16 == 0, "whole MFMA tiles");
  static constexpr int GROUPS = (BM + BN) / 8;                        // a load fills 8 rows of a stage
  static constexpr int ROW_LOADS = (GROUPS + 7) / 8;                  // per wave and stage; the last may repeat a row group
  static constexpr int LOADS = ROW_LOADS + (SCALED ? 1 : 0);
  // A wave's channels are WN consecutive ones inside one 128-channel scale block, except for BN = 192, where 48 consecutive
  // channels could straddle two blocks: there the wave's channel tile i is channels 64 i + 16 wave .. + 15, so that tile i of
  // every wave lies in the block of channel n0 + 64 i.
  static constexpr bool INTERLEAVED = BN == 192;
  static constexpr int SB = INTERLEAVED ? NT : 1;
  static constexpr int W_STRIDE = INTERLEAVED ? 64 * 128 : 16 * 128;  // bytes between a wave's consecutive channel tiles in a stage
  static constexpr int STAGE_BYTES = (BM + BN) * KSTEP;
  __device__ static int channel(int wave_n, int i) { return INTERLEAVED ? i * 64 + wave_n * 16 : wave_n * WN + i * 16; }
};

// One BM x BN output tile at (m0, n0), K blocks of split `split`, by the whole workgroup.
// AR_UE8M0: p.sa / p.sb point to packed exponent words: token word (m, kw) at sa[kw * sa_sk + m], channel word (n, kw) at
// sb[kw * sb_sk + n * sb_sn], byte kb & 3 of word kb >> 2 belongs to K block kb.
template <Arith AR, int BM, int BN, bool SPLIT, int S, bool STREAM, bool ROTATES, bool RAGGED = false>
__device__ __forceinline__ void dma_tile(const GemmParams& p, int m0, int n0, int split) {
  using T = TileShape<AR, BM, BN>;
  static_assert(!RAGGED || ((AR == AR_UNIT || AR == AR_INT8) && !SPLIT && !ROTATES), "the last K block is multiplied last");
  static_assert(S >= 3 && S * (T::STAGE_BYTES + BM * 4) <= 160 * 1024, "the stages must fit the CU's LDS");
  constexpr int MT = T::MT, NT = T::NT, SB = T::SB, LOADS = T::LOADS, WM = T::WM;
  using AccT = typename std::conditional<AR == AR_INT8, int, float>::type;
  typedef AccT acc4 __attribute__((ext_vector_type(4)));
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave / T::WAVES_N, wave_n = wave % T::WAVES_N;
  const int l16 = lane & 15, q = lane >> 4;
  const int kb_begin = split * p.kb_per_split;
  const int nkb = min(p.kb_total, kb_begin + p.kb_per_split) - kb_begin;
  const int kb_last = kb_begin + nkb - 1;

  // the stages: tile rows (0..BM-1 tokens, then channels) and the tile's BM token scales
  __shared__ __attribute__((aligned(1024))) uint8_t t_stage[S * T::STAGE_BYTES];
  __shared__ __attribute__((aligned(256))) float t_scale[S * BM];

  // ---- loader: lane's byte offset from the matrix base for each of its rows (rows clamped); lands swizzled by (row & 7)
  uint32_t goff[T::ROW_LOADS];
  {
    const int lrow = lane >> 3;
    const int chunk_byte = ((lane & 7) ^ lrow) * 16;
#pragma unroll
    for (int i = 0; i < T::ROW_LOADS; ++i) {
      const int row = min(i * 8 + wave, T::GROUPS - 1) * 8 + lrow;
      goff[i] = row < BM ? (uint32_t)((int64_t)min(m0 + row, p.M - 1) * p.lda + chunk_byte)
                         : (uint32_t)((int64_t)min(n0 + row - BM, p.N - 1) * p.ldb + chunk_byte);
    }
  }
  const int tail = p.K - (p.kb_total - 1) * KSTEP;  // bytes of the last K block
  const uint32_t past_end = RAGGED ? (uint32_t)max((((lane & 7) ^ (lane >> 3)) - (tail / 16 - 1)) * 16, 0) : 0u;  // of it, where its row ends
  const int last_group = __builtin_amdgcn_readfirstlane(min((T::ROW_LOADS - 1) * 8 + wave, T::GROUPS - 1));
  // matrix of the wave's row group in the load that covers both kinds of rows (BM not a multiple of 64)
  const bool mixed_tokens = __builtin_amdgcn_readfirstlane(BM / 64 * 8 + wave < BM / 8);
  const uint8_t* mixed_base = mixed_tokens ? p.a : p.b;
  // every wave fetches BM / 8 token scales per K block, four per lane; quads past M refetch the last valid one
  const uint32_t sa_off = (uint32_t)min(m0 + wave * (BM / 8) + min(lane, BM / 32 - 1) * 4, (p.M - 1) & ~3) * 4u;
  // The K loop may start in the middle (the sum is the same products in another order): block k of the loop is block
  // (k + rotation) % nkb of the range.  See rotates_k.
  const int rotation = ROTATES && p.rotate_k ? __builtin_amdgcn_readfirstlane((n0 / BN) % nkb) : 0;
  auto block_of = [&](int kb) {
    kb = min(kb, kb_last) + rotation;
    if (!ROTATES) return kb;
    return kb > kb_last ? kb - nkb : kb;
  };
  // Load number i of K block kb (< ROW_LOADS: tile rows; then the token scales) into stage `st`.  The statements write m0; it
  // cannot be listed as a clobber (the compiler reserves the register), and no compiler-managed use of m0 lies between them
  // and the next statement that sets it.
  auto issue = [&](int i, int st, int kb) {
    kb = block_of(kb);
    if (i < T::ROW_LOADS) {
      // wave-uniform: the row group (the last load's may be one another wave fetches too) and its matrix
      const int group = i * 8 + 8 <= T::GROUPS ? i * 8 + wave : last_group;
      const uint8_t* base = (i * 8 + 8 <= BM / 8 ? p.a : i * 8 >= BM / 8 ? p.b : mixed_base) + (uint64_t)kb * KSTEP;
      asm volatile("" : "+s"(base));
      const uint32_t off = RAGGED ? goff[i] - (kb == kb_last ? past_end : 0u) : goff[i];
      const uint32_t lds_addr = (uint32_t)(uintptr_t)(lptr_t)t_stage + (uint32_t)(st * T::STAGE_BYTES + group * 8 * KSTEP);
      if (STREAM && i * 8 >= BM / 8)  // (weight rows only)
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off), "s"(base), "s"(lds_addr) : "memory");
      else
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_addr) : "memory");
    } else if constexpr (T::SCALED) {
      // BM / 32 lanes fetch 16 bytes each (a 4-byte-per-lane load in this stream costs far more than its size).  exec is
      // narrowed and restored inside the statement.  Packed exponents: one row of words per four K blocks, fetched again for
      // each of the four (the load count per K block stays constant).
      const float* sbase = p.sa + (int64_t)(AR == AR_UE8M0 ? kb >> 2 : kb) * p.sa_sk;  // wave-uniform
      asm volatile("" : "+s"(sbase));
      const uint32_t lds_addr = (uint32_t)(uintptr_t)(lptr_t)t_scale + (uint32_t)(st * BM + wave * (BM / 8)) * 4u;
      uint64_t saved;
      asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_mov_b32 m0, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, %0"
                   : "=&s"(saved) : "v"(sa_off), "s"(sbase), "s"(lds_addr), "n"((1 << (BM / 32)) - 1) : "memory");
    }
  };

  // ---- fragment addresses inside a stage.  Lane quarter q takes the 16-byte chunks q and q + 4 of a row (full LDS rate).
  uint32_t tok_off[2], ch_off[2];
  {
    const int trow = wave_m * WM + l16, crow = BM + T::channel(wave_n, 0) + l16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      tok_off[h] = trow * KSTEP + (((q + 4 * h) ^ (trow & 7)) << 4);
      ch_off[h] = crow * KSTEP + (((q + 4 * h) ^ (crow & 7)) << 4);
    }
  }
  const uint32_t sc_off = (wave_m * WM + l16) * 4;
  cfloat_ptr sb_ptr[SB];  // the wave's (channel tile's) row of weight-block scales
  if constexpr (T::SCALED) {
#pragma unroll
    for (int b = 0; b < SB; ++b) {
      const int first = min(n0 + T::channel(wave_n, b), p.N - 1);
      sb_ptr[b] = (cfloat_ptr)(p.sb + (int64_t)__builtin_amdgcn_readfirstlane(AR == AR_UE8M0 ? first : first / 128) * p.sb_sn);
    }
  }
  float sbv[SB];  // scales (words) of the block to be multiplied next
  auto load_sb = [&](int kb) {
    if constexpr (T::SCALED) {
      kb = block_of(kb);
#pragma unroll
      for (int b = 0; b < SB; ++b) sbv[b] = sb_ptr[b][(int64_t)(AR == AR_UE8M0 ? kb >> 2 : kb) * p.sb_sk];
    }
  };

  acc4 acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = acc4{0, 0, 0, 0};

  // two sets of fragments and token scales
  Frag w[2][NT], tok[2][MT];
  float tsc[2][MT];
  constexpr int READS = 2 * (NT + MT);
  // read number r of a block out of stage `st` into set `set`: token tile 0, the channel tiles, the other token tiles
  auto read = [&](int r, int set, lds_cptr st, lds_cptr sc) {
    const int f = r >> 1, h = r & 1;
    if (f >= 1 && f <= NT) {
      const u32x4 v = lds16(st + ch_off[h], (f - 1) * T::W_STRIDE);
      if (h == 0) w[set][f - 1].lo = v;
      else w[set][f - 1].hi = v;
    } else {
      const int j = f == 0 ? 0 : f - NT;
      const u32x4 v = lds16(st + tok_off[h], j * 2048);
      if (h == 0) tok[set][j].lo = v;
      else tok[set][j].hi = v;
      if (T::SCALED && h == 1) tsc[set][j] = lds_f32(sc + sc_off, j * 64);
    }
  };
  auto stage_at = [&](int st) { return (lds_cptr)t_stage + st * T::STAGE_BYTES; };
  auto scales_at = [&](int st) { return (lds_cptr) reinterpret_cast<uint8_t*>(t_scale) + st * BM * 4; };

  // AR_F32: a product is promoted (acc += product * scale) behind the second MFMA after its own, where its result needs no wait
  // states any more; the last two products of a block are promoted in the next one.
  v4f pend[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
  float pend_scale[2] = {0.f, 0.f};
  auto promote = [&](int t, const v4f& product, float scale) {
    const int j = t / NT, i = t % NT;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[i][j][v] = fmaf(product[v], scale, acc[i][j][v]);
  };

  // Multiplies block k out of set CUR while reading block k + 1 (in stage st_next) into the other set and, with FILL, issuing
  // block k + S into st_fill, the stage block k has just left.
  auto block = [&](auto cur_c, auto fill_c, int k, int st_next, int st_fill) {
    constexpr int CUR = decltype(cur_c)::value, NXT = 1 - CUR;
    constexpr bool FILL = decltype(fill_c)::value;
    const int kb = kb_begin + k;
    const lds_cptr nst = stage_at(st_next), nsc = scales_at(st_next);
    float sc[MT][SB];
    int w_exp[SB];
    if constexpr (AR == AR_F32) {
#pragma unroll
      for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int b = 0; b < SB; ++b) sc[j][b] = tsc[CUR][j] * sbv[b];
    } else if constexpr (AR == AR_UE8M0) {
      const int shift = (block_of(kb) & 3) * 8;
#pragma unroll
      for (int b = 0; b < SB; ++b) w_exp[b] = in_vgpr((int)(__float_as_uint(sbv[b]) >> shift));
#pragma unroll
      for (int j = 0; j < MT; ++j) sc[j][0] = __uint_as_float(__float_as_uint(tsc[CUR][j]) >> shift);
    }
    if constexpr (RAGGED && !FILL) {  // (the last block is among those that request nothing any more)
      const int valid = kb == kb_last ? tail : KSTEP;
      const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        if (16 * q >= valid) tok[CUR][j].lo = z;
        if (64 + 16 * q >= valid) tok[CUR][j].hi = z;
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // the waits for this block's scales come before the scalar load of the next one's
    load_sb(kb + 1);
    __builtin_amdgcn_sched_barrier(0);
    // the reads go out over the first three quarters of the steps, so that the last ones have returned at the barrier
    constexpr int LPS = (LOADS + T::STEPS - 1) / T::STEPS;  // loads per step
    constexpr int PER = (READS * 4 + T::STEPS * 3 - 1) / (T::STEPS * 3);
    v4f part[3];
#pragma unroll
    for (int t = 0; t < T::STEPS; ++t) {
      const int j = t / NT, i = t % NT;
      if constexpr (AR == AR_F32) {
        part[t % 3] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(as_v8i(w[CUR][i]), as_v8i(tok[CUR][j]), v4f{0.f, 0.f, 0.f, 0.f},
                                                                       0, 0, 0, 0, 0, 0);
      } else if constexpr (AR == AR_UE8M0) {
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(as_v8i(w[CUR][i]), as_v8i(tok[CUR][j]), acc[i][j], 0, 0, 0,
                                                                     w_exp[SB > 1 ? i : 0], 0, (int)__float_as_uint(sc[j][0]));
      } else if constexpr (AR == AR_UNIT) {
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(as_v8i(w[CUR][i]), as_v8i(tok[CUR][j]), acc[i][j], 0, 0, 0, 0, 0, 0);
      } else {
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(as_v4i(w[CUR][i].lo), as_v4i(tok[CUR][j].lo), acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(as_v4i(w[CUR][i].hi), as_v4i(tok[CUR][j].hi), acc[i][j], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);  // the MFMA goes first; the rest of the step runs in its shadow
#pragma unroll
      for (int r = t * PER; r < (t + 1) * PER; ++r)
        if (r < READS) read(r, NXT, nst, nsc);
#pragma unroll
      for (int l = t * LPS; l < (t + 1) * LPS; ++l)
        if (FILL && l < LOADS) issue(l, st_fill, kb + S);
      if constexpr (AR == AR_F32) {
        if (t < 2) promote(T::STEPS - 2 + t, pend[t], pend_scale[t]);
        else promote(t - 2, part[(t - 2) % 3], sc[(t - 2) / NT][SB > 1 ? (t - 2) % NT : 0]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (AR == AR_F32) {
#pragma unroll
      for (int e = 0; e < 2; ++e) pend[e] = part[(T::STEPS - 2 + e) % 3], pend_scale[e] = sc[MT - 1][SB > 1 ? NT - 2 + e : 0];
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  // everything but the YOUNGER youngest loads has landed, the wave's LDS reads have returned; then the workgroup barrier
#define MI355_TILE_BARRIER(YOUNGER) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER) : "memory")

  // ---- prologue: blocks 0 .. S-1 (clamped) into the stages, the fragments of block 0 into set 0
#pragma unroll
  for (int b = 0; b < S; ++b)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) issue(i, b, kb_begin + b);
  load_sb(kb_begin);
  MI355_TILE_BARRIER((S - 1) * LOADS);
#pragma unroll
  for (int r = 0; r < READS; ++r) read(r, 0, stage_at(0), scales_at(0));

  // ---- blocks that still request one S further on
  const int nmain = max(nkb - S, 0);
  int st = 0;  // stage of block k
  auto next_stage = [](int s) { return s + 1 == S ? 0 : s + 1; };
  int k = 0;
  for (; k + 1 < nmain; k += 2) {
    const int st1 = next_stage(st), st2 = next_stage(st1);
    MI355_TILE_BARRIER((S - 2) * LOADS);
    block(C0{}, std::true_type{}, k, st1, st);
    MI355_TILE_BARRIER((S - 2) * LOADS);
    block(C1{}, std::true_type{}, k + 1, st2, st1);
    st = st2;
  }
  if (k < nmain) {  // an odd one: the next block's fragments move to set 0
    const int st1 = next_stage(st);
    MI355_TILE_BARRIER((S - 2) * LOADS);
    block(C0{}, std::true_type{}, k, st1, st);
#pragma unroll
    for (int i = 0; i < NT; ++i) w[0][i] = w[1][i];
#pragma unroll
    for (int j = 0; j < MT; ++j) tok[0][j] = tok[1][j], tsc[0][j] = tsc[1][j];
    st = st1;
    ++k;
  }
  // ---- the last blocks (up to S): nothing is requested any more, the number of loads in flight counts down.  The last one
  //      reads a stage for nobody.
#pragma unroll
  for (int u = 0; u < S; ++u) {
    if (u < nkb - nmain) {
      const int st1 = next_stage(st);
      MI355_TILE_BARRIER((u < S - 2 ? S - 2 - u : 0) * LOADS);
      if (u & 1) block(C1{}, std::false_type{}, k + u, st1, 0);
      else block(C0{}, std::false_type{}, k + u, st1, 0);
      st = st1;
    }
  }
  if constexpr (AR == AR_F32) promote(T::STEPS - 2, pend[0], pend_scale[0]), promote(T::STEPS - 1, pend[1], pend_scale[1]);
#undef MI355_TILE_BARRIER
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // refetches of a K shorter than the pipeline must not outlive the workgroup's LDS

  // ---- epilogue: lane holds channels n .. n + 3 of token m for each of its MFMA tiles
  if constexpr (SPLIT) {
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const int m = m0 + wave_m * WM + j * 16 + l16;
      if (m >= p.M) continue;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int n = n0 + T::channel(wave_n, i) + 4 * q;
        if (n >= p.N) continue;  // (N % 4 == 0: all four are in)
        *reinterpret_cast<acc4*>(reinterpret_cast<AccT*>(p.ws) + ((int64_t)split * p.M + m) * p.N + n) = acc[i][j];
      }
    }
  } else {
    if constexpr (AR == AR_INT8) {
      if (p.out_dtype == MI355_I32) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          const int m = m0 + wave_m * WM + j * 16 + l16;
          if (m >= p.M) continue;
#pragma unroll
          for (int i = 0; i < NT; ++i) {
            const int n = n0 + T::channel(wave_n, i) + 4 * q;
            int* o = reinterpret_cast<int*>(p.out) + (int64_t)m * p.ldo + n;
#pragma unroll
            for (int v = 0; v < 4; ++v)
              if (n + v < p.N) o[v] = acc[i][j][v];
          }
        }
        return;
      }
    }
    constexpr OutScale OS = AR == AR_INT8 ? OUT_INT8 : AR == AR_UNIT ? OUT_ROW_COL : OUT_PLAIN;
    static_assert(BM * BN * 2 <= S * T::STAGE_BYTES, "the output tile fits the stages");
    const int row0 = wave_m * WM + l16;
    if (out_tile_ok<OS>(p)) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave's loads have landed: the stages are free
      out_tile_put<OS, BN, NT, MT>(p, t_stage, m0, n0, row0, q, acc, [&](int i) { return T::channel(wave_n, i); });
      __syncthreads();
      out_tile_store<BM, BN>(p, t_stage, m0, n0);
    } else {
      const bool vec_ok = ((p.ldo & 3) == 0) && ((reinterpret_cast<uintptr_t>(p.out) & 15) == 0);
      const float* row_scales = AR == AR_INT8 ? p.sa : p.row_scale;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int n = n0 + T::channel(wave_n, i) + 4 * q;
        const ChannelTerms c = load_channel_terms(p, out_channel_scales<OS>(p), n);
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          const int m = m0 + row0 + j * 16;
          if (m >= p.M || n >= p.N) continue;
          const float token_scale = row_scales ? row_scales[m] : 1.f;
          float r[4];
          if constexpr (AR == AR_INT8) {
            const int a4[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
            int8_apply_terms(p, c, token_scale, a4, r);
          } else {
            r[0] = acc[i][j][0], r[1] = acc[i][j][1], r[2] = acc[i][j][2], r[3] = acc[i][j][3];
            fp8_apply_terms(p, c, token_scale, r);
          }
          store_out4(p.out, p.out_dtype, (int64_t)m * p.ldo + n, r, min(4, p.N - n), vec_ok);
        }
      }
    }
  }
}

// Stages per tile shape: as many as the LDS holds, up to six.  A 64 x 128 tile's three stages take 73.5 KB, so two such
// workgroups share a CU and keep four blocks in flight between them; where a launch has at most one workgroup per CU it runs
// six stages instead.
constexpr int stages_of(int bm, int bn, bool own_cu) {
  return bm + bn == 192 ? (own_cu ? 6 : 3) : bm + bn == 224 ? 5 : bm + bn <= 288 ? 4 : 3;
}

template <Arith AR, int BM, int BN, bool SPLIT, int S, bool STREAM, bool ROTATES, bool RAGGED = false>
__global__ __launch_bounds__(T_THREADS) __attribute__((amdgpu_waves_per_eu(BM + BN == 192 && S == 3 ? 4 : 2))) void gemm_dma_kernel(const GemmParams p) {
  const TileCoord tc = tile_of_block(blockIdx.x, gridDim.x, p.tiles_m, p.tiles_n);
  dma_tile<AR, BM, BN, SPLIT, S, STREAM, ROTATES, RAGGED>(p, tc.tile_m * BM, tc.tile_n * BN, tc.split);
}

template <Arith AR, int BM, int BN>
int launch_dma_tile(GemmParams& p, hipStream_t stream, const char* what) {
  p.tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN - 1) / BN;
  p.rotate_k = p.K % KSTEP == 0 && rotates_k(p.N, p.K, p.ldb);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n * p.splits));
  constexpr int OWN = stages_of(BM, BN, true), SHARED = stages_of(BM, BN, false);
  // (a kernel of its own for K loops that start in the middle: the few instructions more cost a chain of short K blocks 5 %, 16 experts of
  // 36 rows, 3840 -> 256, 17.7 / 18.6 us; the streamed one has them, its blocks wait for memory)
  const auto launch = [&](auto split, auto streamed, auto rotates) {
    constexpr bool SPLIT = decltype(split)::value, STREAM = decltype(streamed)::value, ROTATES = decltype(rotates)::value;
    if (OWN != SHARED && (int64_t)p.tiles_m * p.tiles_n * p.splits > NUM_CUS) launch_kernel((gemm_dma_kernel<AR, BM, BN, SPLIT, SHARED, STREAM, ROTATES>), grid, dim3(T_THREADS), 0, stream, p);
    else launch_kernel((gemm_dma_kernel<AR, BM, BN, SPLIT, OWN, STREAM, ROTATES>), grid, dim3(T_THREADS), 0, stream, p);
  };
  const std::true_type yes;
  const std::false_type no;
  if constexpr (AR == AR_UNIT || AR == AR_INT8) {
    if (p.K % KSTEP != 0) {
      const auto launch_ragged = [&](auto streamed) {
        constexpr bool STREAM = decltype(streamed)::value;
        if (OWN != SHARED && (int64_t)p.tiles_m * p.tiles_n > NUM_CUS) launch_kernel((gemm_dma_kernel<AR, BM, BN, false, SHARED, STREAM, false, true>), grid, dim3(T_THREADS), 0, stream, p);
        else launch_kernel((gemm_dma_kernel<AR, BM, BN, false, OWN, STREAM, false, true>), grid, dim3(T_THREADS), 0, stream, p);
      };
      if (p.splits != 1) {
        set_error("%s: the mid-M tile does not split a K of parts of blocks", what);
        return MI355_ERR_UNSUPPORTED;
      }
      if (BM == 64 && streams_weight(p)) launch_ragged(std::integral_constant<bool, BM == 64>{});
      else launch_ragged(no);
      return check_launch(what);
    }
  }
  const auto launch_split = [&](auto split) {
    const std::integral_constant<bool, !decltype(split)::value || BM == 64> may_stream;
    if (may_stream && streams_weight(p)) launch(split, may_stream, yes);
    else if (p.rotate_k) launch(split, no, yes);
    else launch(split, no, no);
  };
  if (p.splits > 1) launch_split(yes);
  else launch_split(no);
  return check_launch(what);
}

// The tile shapes that are built (MID_TILES in gemm_common.h), by height and width.
template <Arith AR, size_t... I>
int launch_dma_tile_of(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what, std::index_sequence<I...>) {
  int rc = MI355_ERR_UNSUPPORTED;
  bool found = false;
  ((found = found || (bm == MID_TILES[I].bm && bn == MID_TILES[I].bn && (rc = launch_dma_tile<AR, MID_TILES[I].bm, MID_TILES[I].bn>(p, stream, what), true))), ...);
  if (!found) set_error("%s: no %d x %d tile is built", what, bm, bn);
  return rc;
}
template <Arith AR>
int launch_dma_tile_of(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_dma_tile_of<AR>(p, bm, bn, stream, what, std::make_index_sequence<sizeof(MID_TILES) / sizeof(MID_TILES[0])>{});
}

}  // namespace
}  // namespace mi355
