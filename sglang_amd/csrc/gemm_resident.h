// GEMMs of short K and many tokens for gfx950: the weight stays in registers, the tokens stream past it and the results leave from
// registers while the next tokens are multiplied.  256 channels per workgroup, K = 256 .. 768.
//
// A tile that is computed and then stored spends as long on its result as on its products when K is short: K = 512 -> N = 32768 at 3001
// tokens took 87 us on the 256 x 256 two-phase tile, half of it the result's 197 MB on their way out with the matrix pipe idle.  Stores
// cannot be overlapped with the next operands by the wave that waits for those (vmcnt counts loads and stores together, and only loads
// complete in order), so here other waves load:
//   waves 0..7   (two per SIMD) hold 32 channels x K of the weight in registers for the whole launch; they read the tokens from LDS,
//                multiply, convert and store: they never wait for memory;
//   waves 8, 9   request tokens and token scales S - 1 steps ahead, straight into LDS, and wait for them.
// A step is two half steps of 32 tokens (16 where the registers hold no more beside the weight) with accumulators of their own: one half's
// results leave behind the first products of the other.  One barrier per step says that the step after the next has landed and that the
// last one's stage is free; a wave has its first fragments of a step in registers when it passes it.
// A lane's results are eight consecutive channels of a token, because the weight's rows are dealt to the two channel tiles of a wave in
// fours (channel 8 q + 4 c + v is row 4 q + v of tile c): 16-byte stores without a pass through LDS.
// Tokens are read from L2 once per 256 channels (16 bytes a cycle and CU).
// What bounds it: the products and their promotion, about as many cycles of the vector unit as of the matrix pipe, then the stores (512 -> 32768 at 3001
// tokens takes 55 us, packed exponents 62, where the results go to memory).  A result costs a conversion and a sixteenth of a store: the loop is a kernel of its own for each output
// type, with and without a bias, written through or not, the stores are buffer stores whose range check drops what does not exist, and their
// addresses advance in scalar registers.  With these choices and checks in the loop every half step ran through a dozen branches and 50 vector
// instructions beside the promotion's 64, and the compiler moved products across the branches; us of the GPU, before / now, 3001 tokens 512 -> 32768 in a loop on
// one set of buffers: FP8 56.5 / 53, packed exponents 51 / 46, epilogue scales 58 / 50, INT8 63 / 51; 36 random linears 0.91.  One choice alone as a branch in the
// loop, 80 random linears: the bias packed exponents 1.13 (of K = 640 and 768 1.9 to 3.7, spilled), the others, which have one scheme with them, 1.00; writing
// through packed exponents 1.015 (20 of 17 to 120 MB) and 1.02 (20 of more than 128 MB), whose products are sunk behind it, the others 1.00.
// Whole linears, us, two-phase tile / this:
//   block FP8 3001 tokens 512 -> 32768 89.9 / 73.9, 2310 tokens 256 -> 32768 56.2 / 36.3, 1966 tokens 640 -> 16384 43.1 / 31.2;
//   packed exponents 1609 tokens 512 -> 32768 63.6 / 36.6;  per token FP8 820 tokens 512 -> 32768 37.8 / 24.3;  INT8 952 tokens 640 -> 32768 38.6 / 29.1;
//   K = 768, the longest whose weight is not spilled (153 to 165 registers of 168; 896 is), whatever ran before / this: block FP8 611 tokens -> 13312 19.0 / 15.2,
//   1706 tokens -> 24576 60.0 / 53.5, packed exponents 1493 tokens -> 7296 20.9 / 17.1, per token FP8 827 tokens -> 24576 32.5 / 24.0, INT8 1308 tokens ->
//   14848 34.8 / 25.6; 40 random linears 0.83.  There the stores take a fifth of the time, the token loads 3 % (each left out).
// Tried: store waves with the results in LDS between (75), fragments two blocks ahead (equal), four waves of 64 channels (62), two smaller
// workgroups a CU (81), all 55 here before, us for the first of those shapes in a loop on one set of buffers; the two waves of a SIMD storing at different
// products (53 / 55); K = 640 and 768 with fragments two blocks ahead (equal), and with nontemporal stores (0.92 to 0.95 alone where every call has
// results of its own, 1.03 to 1.04 in a loop on the same ones and with a quantizer that reads them).
#pragma once

#include "gemm_dma_tile.h"

namespace mi355 {
namespace {

constexpr int RS_BN = RESIDENT_CHANNELS, RS_COMPUTE = 8, RS_LOAD = 2, RS_WEIGHT_SLOTS = 3, RS_CT = 2;
constexpr int RS_THREADS = 64 * (RS_COMPUTE + RS_LOAD);

// Tokens of a half step.  With a bias the unscaled kinds' epilogue takes twelve registers more, which would be spilled beside K = 512 and 32 tokens (a
// reload waits for every store in flight): 32 random linears, half steps of 32 / of 16: per-token FP8 1.10 in a graph and 1.11 eager, INT8 1.01 and 1.01.  (INT8
// of K = 512 spills a register or two, block FP8 of K = 512 with a bias and results beyond 128 MB four, outside the loop.)  The
// choice of ranges and the plan go by the steps without a bias, which take 1 to 3 % less time.
template <Arith AR, int KB, bool BIAS>
constexpr int rs_half_step() { return BIAS && KB == 4 && (AR == AR_UNIT || AR == AR_INT8) ? 16 : resident_half_step(AR == AR_UE8M0, KB); }

template <Arith AR, int KB, bool BF16, bool BIAS, bool THROUGH>
__global__ __launch_bounds__(RS_THREADS) __attribute__((amdgpu_waves_per_eu(3))) void resident_kernel(const GemmParams p, const int ranges, const int steps_per_range) {
  constexpr bool SCALED = AR == AR_F32 || AR == AR_UE8M0;
  constexpr int HALF = rs_half_step<AR, KB, BIAS>(), TS = 2 * HALF, TT = HALF / 16, CT = RS_CT;  // tokens of a half step, of a step
  constexpr int KBLOCK = TS * KSTEP, STAGE = KB * KBLOCK, SCALE_BYTES = 1024 * TS / 32;
  constexpr int LOADS = KB * (TS / 8) / RS_LOAD + (SCALED ? TS / 32 : 1);  // per load wave and step: tokens, and the step's scales
  constexpr int SLOT = CT * 16 * KSTEP, STAGING = RS_COMPUTE * RS_WEIGHT_SLOTS * SLOT;  // the weight's way into the registers
  constexpr int FIT = 160 * 1024 / (STAGE + SCALE_BYTES), S = FIT > 8 ? 8 : FIT;
  constexpr int FIRST = 1;  // stages that are filled beside the staging area
  constexpr int BYTES = S * STAGE > FIRST * STAGE + STAGING ? S * STAGE : FIRST * STAGE + STAGING;
  static_assert(KB >= 2 && KB <= RESIDENT_MAX_KBLOCKS && S >= 4 && BYTES + S * SCALE_BYTES <= 160 * 1024, "built for these");
  static_assert((S - 3) * LOADS < 64, "vmcnt");
  using AccT = typename std::conditional<AR == AR_INT8, int, float>::type;
  typedef AccT acc4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(1024))) uint8_t mem[BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t scales[S * SCALE_BYTES];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // consecutive workgroups of an XCD take the token ranges of the same channels
  int bid = blockIdx.x;
  const int per_xcd = (int)gridDim.x >> 3;
  if (bid < per_xcd * 8) bid = (bid & 7) * per_xcd + (bid >> 3);
  const int slice = __builtin_amdgcn_readfirstlane(bid / ranges);  // (the division is done by vector instructions)
  const int n0 = slice * RS_BN, m_begin = (bid - slice * ranges) * steps_per_range * TS;
  const int steps = min(steps_per_range, (p.M - m_begin + TS - 1) / TS);
#define MI355_RS_BARRIER() asm volatile("s_barrier" ::: "memory")

  if (wave >= RS_COMPUTE) {
    // ================= load waves =================
    const int lw = wave - RS_COMPUTE;
    constexpr int GROUPS = TS / 8 / RS_LOAD;  // 8-row groups of a wave
    const int chunk_byte = ((lane & 7) ^ (lane >> 3)) * 16;
    const float* row_scales = AR == AR_INT8 ? p.sa : p.row_scale;
    auto issue = [&](int i, int st) {
      const int m0 = m_begin + i * TS;
      const uint32_t stage = (uint32_t)(uintptr_t)(lptr_t)mem + (uint32_t)(st * STAGE);
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
        const int row = (lw * GROUPS + g) * 8;
        const uint32_t off = (uint32_t)((int64_t)min(m0 + row + (lane >> 3), p.M - 1) * p.lda + chunk_byte);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          const uint8_t* base = p.a + kb * KSTEP;
          const uint32_t dst = stage + (uint32_t)(kb * KBLOCK + row * KSTEP);
          asm volatile("" : "+s"(base));
          asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(dst) : "memory");
        }
      }
      // Both load waves fetch the scales, the same values to the same place: their load counts stay equal.
      const uint32_t dst = (uint32_t)(uintptr_t)(lptr_t)scales + (uint32_t)(st * SCALE_BYTES);
      if constexpr (SCALED) {
        // eight lanes fetch 32 scales (exponent words) of a K block (of four); rows and quads past the end repeat the last
        constexpr int ROWS = AR == AR_UE8M0 ? (KB + 3) / 4 : KB;
#pragma unroll
        for (int h = 0; h < TS / 32; ++h) {
          const float* src = p.sa + (int64_t)min(lane >> 3, ROWS - 1) * p.sa_sk + min(m0 + h * 32 + (lane & 7) * 4, (p.M - 1) & ~3);
          asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(dst + h * 1024) : "memory");
        }
      } else {
        const float* src = row_scales + min(m0 + lane, p.M - 1);
        asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(dst) : "memory");
      }
    };
    int issued = 0;
    for (; issued < min(steps, FIRST); ++issued) issue(issued, issued);
    MI355_RS_BARRIER();  // weight in registers: the other stages are free
    for (; issued < min(steps, S - 1); ++issued) issue(issued, issued);
    if (steps >= S - 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 3) * LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    MI355_RS_BARRIER();  // steps 0 and 1 have landed
    int st = S - 1;  // stage of step i + S - 1, which is that of step i - 1
    for (int i = 0; i + 1 < steps; ++i) {
      if (i + S - 1 < steps) {
        issue(i + S - 1, st);
        st = st + 1 == S ? 0 : st + 1;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 3) * LOADS) : "memory");  // step i + 2 has landed
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      MI355_RS_BARRIER();
    }
    return;
  }

  // ================= compute waves =================
  const int l16 = lane & 15, q = lane >> 4;
  const int n_wave = n0 + wave * (16 * CT);
  const uint32_t off[2] = {(uint32_t)(l16 * KSTEP + ((q ^ (l16 & 7)) << 4)), (uint32_t)(l16 * KSTEP + (((q + 4) ^ (l16 & 7)) << 4))};

  // ---- the wave's channels x K into registers, through slots of its own (whole 128-byte lines; fetched in the MFMA's layout the same
  //      bytes come at a third of the rate)
  Frag w[KB][CT];
  {
    constexpr int WL = CT * 2;  // loads of a K block
    const uint32_t slots = (uint32_t)(FIRST * STAGE + wave * RS_WEIGHT_SLOTS * SLOT);
    uint32_t goff[WL];
#pragma unroll
    for (int g = 0; g < WL; ++g)
      goff[g] = (uint32_t)((int64_t)min(n_wave + g * 8 + (lane >> 3), p.N - 1) * p.ldb + ((lane & 7) ^ (lane >> 3)) * 16);
    auto issue = [&](int kb) {
      const uint8_t* base = p.b + kb * KSTEP;
      asm volatile("" : "+s"(base));
#pragma unroll
      for (int g = 0; g < WL; ++g) {
        const uint32_t dst = (uint32_t)(uintptr_t)(lptr_t)mem + slots + (uint32_t)((kb % RS_WEIGHT_SLOTS) * SLOT + g * 1024);
        asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(goff[g]), "s"(base), "s"(dst) : "memory");
      }
    };
#pragma unroll
    for (int kb = 0; kb < RS_WEIGHT_SLOTS && kb < KB; ++kb) issue(kb);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int younger = min(KB - 1 - kb, RS_WEIGHT_SLOTS - 1);
      if (younger == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * WL) : "memory");
      else if (younger == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WL) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const lds_cptr slot = (lds_cptr)mem + slots + (kb % RS_WEIGHT_SLOTS) * SLOT;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const int row = 8 * (l16 >> 2) + 4 * c + (l16 & 3);  // of the wave's channels
        w[kb][c].lo = lds16(slot + row * KSTEP + ((q ^ (row & 7)) << 4), 0);
        w[kb][c].hi = lds16(slot + row * KSTEP + (((q + 4) ^ (row & 7)) << 4), 0);
      }
      if (kb + RS_WEIGHT_SLOTS < KB) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(kb + RS_WEIGHT_SLOTS);
      }
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  MI355_RS_BARRIER();  // weight in registers: its staging area is free

  // ---- what does not change from step to step
  float sb[KB];
  int w_exp[KB];
  if constexpr (SCALED) {
    const int first = min(n_wave, p.N - 1);
    const cfloat_ptr row = (cfloat_ptr)(p.sb + (int64_t)__builtin_amdgcn_readfirstlane(AR == AR_UE8M0 ? first : first / 128) * p.sb_sn);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const float v = row[(int64_t)(AR == AR_UE8M0 ? kb >> 2 : kb) * p.sb_sk];
      if constexpr (AR == AR_UE8M0) w_exp[kb] = in_vgpr((int)(__float_as_uint(v) >> ((kb & 3) * 8)));
      else sb[kb] = v;
    }
  }
  const int n = n_wave + 8 * q;  // the lane's eight channels (whole: N % 8 == 0)
  v4f cs[CT];
  u32x2 hb[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int nc = min(n + 4 * c, p.N - 4);  // (channels past N are never stored)
    if constexpr (!SCALED) cs[c] = *reinterpret_cast<const v4f*>((AR == AR_INT8 ? p.sb : p.col_scale) + nc);
    hb[c] = p.bias ? *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(p.bias) + nc) : u32x2{0u, 0u};
  }
  // Two half steps, each with accumulators of its own: one's results are converted and stored while the other's products are formed.
  acc4 acc[2][CT][TT] = {};
  float row_ts[2][TT] = {};
  Frag tok[2][TT];
  float ts[2][TT], sc[2][TT] = {};
  v4f part[4] = {};
  constexpr int LAST = KB * TT * CT;  // products of a half step
  // Behind which product the half step before this one starts to leave: soon, or, where it has 32 tokens and its results are not written through, behind the
  // last ones.  80 linears, graph, late / soon: results beyond 128 MB of K = 256 and 384 0.98, packed exponents 0.92, of K = 512 0.95 (3001 tokens -> 32768 block FP8
  // 79 / 72 us, INT8 74 / 69); of half steps of 16 tokens 1.00; results that are written through 1.02.  Left soon, packed exponents of K = 256 and 384 took up to
  // 1.10 of the time of the loop with all choices in it, whose stores its branches held up.
  constexpr int EMIT = !THROUGH && TT == 2 ? LAST - TT : 2;
  static_assert(LAST % 2 == 0, "the ring of products continues from step to step");
  auto ring = [](int h, int s) { return (h * LAST + s) & 3; };

  // Where the results of token tile t of a half step go, from its first row on: buffer stores, whose range check drops the rows past the
  // last token and, by an offset past every range, the lanes past the last channel.
  uint32_t at[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t) at[t] = n < p.N ? (uint32_t)((t * 16 + l16) * (int)p.ldo + n) * 2u : 0x80000000u;
  const auto rows_of = [&](int m0, bool any) {
    const int rows = any ? max(min(p.M - m0, HALF), 0) : 0;
    const uint64_t base = reinterpret_cast<uint64_t>(p.out) + (uint64_t)((int64_t)(any ? m0 : m_begin) * p.ldo * 2);
    const uint64_t scalar = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(base >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(scalar), (short)0, __builtin_amdgcn_readfirstlane(rows * (int)p.ldo * 2), 0x00027000);
  };
  // fragments and scales of K block kb of half step h (in stage st) into set `set`
  auto read = [&](int set, int st, int h, int kb) __attribute__((always_inline)) {
    const lds_cptr at = (lds_cptr)mem + st * STAGE, sc_at = (lds_cptr)scales + st * SCALE_BYTES + l16 * 4;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      tok[set][t].lo = lds16(at + off[0], kb * KBLOCK + (h * TT + t) * 2048);
      tok[set][t].hi = lds16(at + off[1], kb * KBLOCK + (h * TT + t) * 2048);
      constexpr int PER = 32 / 16;  // token tiles of a load of scales
      const int tile = h * TT + t;
      if constexpr (SCALED) ts[set][t] = lds_f32(sc_at, tile / PER * 1024 + ((AR == AR_UE8M0 ? kb >> 2 : kb) * 32 + tile % PER * 16) * 4);
      else if (kb == 0) row_ts[h][t] = lds_f32(sc_at, tile * 64);
    }
  };
  // AR_F32: product s of half step h is promoted behind the second MFMA after its own, where it needs no wait states any more
  auto promote = [&](int h, int s) __attribute__((always_inline)) {
    const int c = s % CT, t = (s / CT) % TT, kb = s / (CT * TT), set = (h * KB + kb) & 1;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[h][c][t][v] = kb == 0 ? part[ring(h, s)][v] * sc[set][t] : fmaf(part[ring(h, s)][v], sc[set][t], acc[h][c][t][v]);
    asm volatile("" : "+v"(acc[h][c][t]));  // here, in the shadow of the products (the compiler collects them behind the barrier otherwise)
  };
  MI355_RS_BARRIER();  // steps 0 and 1 have landed
  read(0, 0, 0, 0);

  // eight channels of token tile t of half step h, whose tokens have the scale `row`, converted and stored
  const auto emit = [&](int h, int t, float row, __amdgpu_buffer_rsrc_t to) __attribute__((always_inline)) {
    uint32_t word[2 * CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      float r[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {  // separately rounded steps, as in out_tile_put
        if constexpr (AR == AR_INT8) r[v] = mul_rn((float)acc[h][c][t][v], mul_rn(cs[c][v], row));
        else if constexpr (AR == AR_UNIT) r[v] = mul_rn(row, mul_rn(cs[c][v], acc[h][c][t][v]));
        else r[v] = acc[h][c][t][v];
      }
      if constexpr (BIAS) {
        const uint32_t b[4] = {hb[c].x & 0xffffu, hb[c].x >> 16, hb[c].y & 0xffffu, hb[c].y >> 16};
        if constexpr (SCALED) {
          float rounded[4] = {r[0], r[1], r[2], r[3]};
          round_to_16_bits<BF16>(rounded);
#pragma unroll
          for (int v = 0; v < 4; ++v) r[v] = p.bias_rounded ? rounded[v] : r[v];  // (a selection: no branch may part the products)
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) r[v] = add_rn(r[v], BF16 ? bf16_bits_to_f32(b[v]) : f16_bits_to_f32(b[v]));
      }
      word[2 * c] = BF16 ? pack_bf16x2(r[0], r[1]) : pack_f16x2(r[0], r[1]);
      word[2 * c + 1] = BF16 ? pack_bf16x2(r[2], r[3]) : pack_f16x2(r[2], r[3]);
    }
    const u32x4 v = {word[0], word[1], word[2], word[3]};
    __builtin_amdgcn_raw_buffer_store_b128(v, to, at[t], 0, THROUGH ? 16 : 0);  // (16: sc1)
  };
  int st = 0;
  for (int i = 0; i < steps; ++i) {
    const int st_next = st + 1 == S ? 0 : st + 1;
    const int m0 = m_begin + i * TS;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const auto to = rows_of(h == 1 ? m0 : m0 - HALF, h == 1 || i > 0);  // (none before the first half step)
      float row_before[TT];  // (the last block's read brings the scales of the half step after this one)
#pragma unroll
      for (int t = 0; t < TT; ++t) row_before[t] = row_ts[h ^ 1][t];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const int set = (h * KB + kb) & 1;  // fragment sets alternate
        if (kb + 1 < KB) read(set ^ 1, st, h, kb + 1);
        else if (h == 0) read(set ^ 1, st, 1, 0);
        else read(set ^ 1, st_next, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            const int s = (kb * TT + t) * CT + c;
            const acc4 zero = {0, 0, 0, 0};
            const acc4 in = kb == 0 ? zero : acc[h][c][t];
            if constexpr (AR == AR_F32) {
              if (c == 0) sc[set][t] = ts[set][t] * sb[kb];
              part[ring(h, s)] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(as_v8i(w[kb][c]), as_v8i(tok[set][t]), v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
              __builtin_amdgcn_sched_barrier(0);
              if (s >= 2) promote(h, s - 2);
              else promote(h ^ 1, LAST - 2 + s);
            } else if constexpr (AR == AR_UE8M0) {
              acc[h][c][t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(as_v8i(w[kb][c]), as_v8i(tok[set][t]), in, 0, 0, 0, w_exp[kb], 0,
                                                                           (int)(__float_as_uint(ts[set][t]) >> ((kb & 3) * 8)));
            } else if constexpr (AR == AR_UNIT) {
              acc[h][c][t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(as_v8i(w[kb][c]), as_v8i(tok[set][t]), in, 0, 0, 0, 0, 0, 0);
            } else {
              acc[h][c][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(as_v4i(w[kb][c].lo), as_v4i(tok[set][t].lo), in, 0, 0, 0);
              acc[h][c][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(as_v4i(w[kb][c].hi), as_v4i(tok[set][t].hi), acc[h][c][t], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (s >= EMIT && s < EMIT + TT) emit(h ^ 1, s - EMIT, row_before[s - EMIT], to);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
    }
    if constexpr (AR != AR_F32) {
#pragma unroll
      for (int e = 0; e < 2 * CT * TT; ++e) asm volatile("" : "+v"(acc[e / (CT * TT)][e / TT % CT][e % TT]));  // in front of the barrier (they would be sunk behind it)
    }
    st = st_next;
    if (i + 1 < steps) MI355_RS_BARRIER();  // the next step but one has landed; this step's stage is free
  }
  if constexpr (AR == AR_F32) promote(1, LAST - 2), promote(1, LAST - 1);
  const auto last = rows_of(m_begin + steps * TS - HALF, true);
#pragma unroll
  for (int t = 0; t < TT; ++t) emit(1, t, row_ts[1][t], last);
#undef MI355_RS_BARRIER
}

template <Arith AR, int KB>
int launch_resident_inst(const GemmParams& p, int ranges, hipStream_t stream, const char* what) {
  const int per_step = 2 * (p.bias != nullptr ? rs_half_step<AR, KB, true>() : rs_half_step<AR, KB, false>()), all = (p.M + per_step - 1) / per_step, steps = (all + ranges - 1) / ranges;
  ranges = (all + steps - 1) / steps;  // none without tokens
  const int slices = (p.N + RS_BN - 1) / RS_BN;
  const auto launch = [&](auto bf16, auto bias, auto through) {
    launch_kernel((resident_kernel<AR, KB, decltype(bf16)::value, decltype(bias)::value, decltype(through)::value>), dim3((unsigned)(slices * ranges)),
                  dim3(RS_THREADS), 0, stream, p, ranges, steps);
  };
  const std::true_type yes;
  const std::false_type no;
  const auto launch_through = [&](auto bf16, auto bias) { p.write_through ? launch(bf16, bias, yes) : launch(bf16, bias, no); };
  const auto launch_bias = [&](auto bf16) { p.bias != nullptr ? launch_through(bf16, yes) : launch_through(bf16, no); };
  p.out_dtype == MI355_BF16 ? launch_bias(yes) : launch_bias(no);
  return check_launch(what);
}
// `ranges`: workgroups that share a slice of 256 channels, each with its own tokens (the last may have fewer).
template <Arith AR>
int launch_resident_of(GemmParams& p, int ranges, hipStream_t stream, const char* what) {
  p.splits = 1;
  switch (p.kb_total) {
    case 2: return launch_resident_inst<AR, 2>(p, ranges, stream, what);
    case 3: return launch_resident_inst<AR, 3>(p, ranges, stream, what);
    case 4: return launch_resident_inst<AR, 4>(p, ranges, stream, what);
    case 5: return launch_resident_inst<AR, 5>(p, ranges, stream, what);
    case 6: return launch_resident_inst<AR, 6>(p, ranges, stream, what);
  }
  set_error("%s: the resident-weight kernel takes K of two to six blocks", what);
  return MI355_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace mi355
