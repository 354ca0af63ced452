// silu(gate) * up fused in front of the 1 x 128 FP8 group quantizer, plain and masked (expert-major) layouts, for gfx950.
//
// What the reference's v2 quantizer does with fuse_silu_and_mul (sgl-kernel/csrc/gemm/per_token_group_quant_8bit_v2.cu:
// :250-392, schedulers :133-238): the input row holds 2 * H values, gate | up; the value that is quantized is
//   v = T( float(T(silu(float(gate)))) * float(up) ),   silu(g) = g / (1 + exp(-g)),   T = the input's 16-bit type,
// then, per group of 128 values, amax = max(1e-10, max |v|), e = ceil(log2(amax / 448)), code = e4m3fn(clamp(v * 2^-e)),
// and the scale leaves as the exponent byte e + 127, four to a 32-bit word, words column-major (token index fastest).
// The reference only builds this combination (column-major packed UE8M0 scales, group 128 in its callers); so does this file.
// Masked layout: x [E, T, 2H], tokens t >= masked_m[e] of expert e are not read; they are left alone, or (zero_rest) written
// as zeros by the same launch, which a caller that hands out the whole tensor otherwise does with two fills in front.
//
// T(silu(g)) is a function of a 16-bit input: it is LOOKED UP.  Evaluated per element (an exp and an IEEE division, ~38
// vector operations per value) the kernel was bound by the vector ALUs at about half of the memory bandwidth; one LDS read
// per value leaves ~10 operations and the kernel bound by HBM.  The two tables (bfloat16, float16: 128 KB each) are
// computed at build time by gen_silu_table.cpp with one fixed sequence of individually rounded fp32 operations - the
// definition the CPU oracle restates, so results are reproducible bit for bit (the reference uses its GPU's approximate
// exp intrinsic and compares its kernels with a tolerance) - and are part of the code object: nothing is initialised at
// run time.  Three forms, chosen by type and number of groups (SQ_NEAR_GROUPS):
//   * ST_WHOLE: 256 workgroups of 1024 threads (one per CU), each with the table copied into LDS (128 of the CU's 160 KB);
//   * ST_NEAR: the copy takes longer than the work where there is little of it, and sixteen waves a CU keep too few loads in
//     flight.  256-thread workgroups with the entries of ordinary bfloat16 magnitudes only (12 KB); a lane with any other gate
//     (zero, huge, infinite, NaN) looks its eight up in the table where it lies.  Costs two more operations a value, which is
//     why the largest inputs take ST_WHOLE;
//   * ST_IN_PLACE: float16 (the same magnitudes would be 76 KB), few groups: every value is looked up where the table lies.
// A 16-lane row of a wave takes a group (8 values per lane: one 16-byte load of gate, one of up, eight lookups, one 8-byte
// store), the loads of the next two groups are requested before the current one is processed.  4 B in and 1 B out per value.
//
// Rows in use are dealt out over the whole launch: every workgroup scans the experts' row counts (they are on the device) and
// walks the list of used rows of all experts with the grid's stride.  With a fixed share of the workgroups per expert the
// fullest expert set the time: 32 experts of 256 rows, half of them used on average, took 17.8 us, the fills 5.5 + 1.8 more.
// The expert of a row is found by bisection of the prefix sums: stepping through them one by one, 256 experts of 16 rows took
// 22.9 us (now 8.9), 256 of 64 rows 49.6 (26.4); 32 of 256 rows 16.0 (12.6 with the near gates in LDS).
#include <algorithm>

#include "common.h"

namespace mi355 {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

__device__ __attribute__((aligned(16))) const uint16_t g_silu_table[2][65536] = {
#include "silu_table.inc"
};

enum SiluTable { ST_IN_PLACE, ST_NEAR, ST_WHOLE };
// The entries of ST_NEAR: bfloat16 gates of 2^-16 <= |gate| < 2^8.  Both signs of a magnitude lie next to each other, so that entry
// r - 2 NEAR_FIRST holds the gate whose bits rotated left by one are r, and one comparison tells whether it is there.
constexpr int NEAR_FIRST = 0x3780, NEAR_COUNT = 24 * 128;

// round a float to T and back
template <int DT>
__device__ __forceinline__ float round_to_t(float v) {
  if constexpr (DT == MI355_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(v));
  return f16_bits_to_f32(f32_to_f16_bits(v));
}
template <int DT>
__device__ __forceinline__ float t_bits_to_f32(uint32_t h) {
  if constexpr (DT == MI355_BF16) return bf16_bits_to_f32(h);
  return f16_bits_to_f32(h);
}

__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true)));
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true)));
  return v;
}

struct SiluQuantParams {
  const void* x;         // [E, T, 2H]
  uint8_t* q;            // [E, T, H]
  uint32_t* s;           // exponent bytes: word (e, t, kw) at e * s_e + kw * s_k + t, byte kg & 3
  const int32_t* masked_m;  // [E] or nullptr (E == 1)
  int64_t T, H;
  int64_t s_e, s_k;      // strides in 32-bit words
  int E, zero_rest;
  int gpr;               // groups per row (H / 128)
  FastDiv div_gpr;
};

constexpr int SQ_MAX_EXPERTS = 1024;           // per launch: the scan of their row counts is one value per thread, at most four
// Which table, by the number of groups.  Measured, us a call (H = 2048, masked with about half of the rows in use), bfloat16,
// near gates / whole table: 8192 groups 4.2 / 5.5, 32768 7.0 / 8.1, 48000 9.4 / 9.8, 65536 11.6 / 11.2, 524288 63.7 / 61.1;
// masked 65536 8.2 / 11.0, 131072 12.6 / 14.9, 524288 44.0 / 45.9.  float16, in place / whole table: 11200 5.5 / 5.6,
// 16384 6.4 / 5.9, 65536 18.9 / 11.2; masked 32768 8.1 / 9.4, 65536 13.2 / 11.0, 131072 20.3 / 15.1.
constexpr int64_t SQ_NEAR_GROUPS = 49152, SQ_NEAR_GROUPS_MASKED = 524288;
constexpr int64_t SQ_IN_PLACE_GROUPS = 12288, SQ_IN_PLACE_GROUPS_MASKED = 32768;
constexpr int SQ_NEAR_WORKGROUPS = 6 * 256;  // six fit a CU by their registers

// Row counts of the experts as prefix sums in LDS: pre[e] = used rows of experts < e, pre[E] = all of them.
template <int THREADS>
__device__ __forceinline__ void scan_rows(const SiluQuantParams& p, int* pre) {
  __shared__ int wave_sum[THREADS / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int base = 0;
  for (int c = 0; c < p.E; c += THREADS) {
    const int e = c + tid;
    const int rows = e < p.E ? (p.masked_m ? min(max(p.masked_m[e], 0), (int)p.T) : (int)p.T) : 0;
    int sum = rows;  // inclusive over the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(sum, d);
      if (lane >= d) sum += up;
    }
    if (lane == 63) wave_sum[wave] = sum;
    __syncthreads();
    int before = base;
    for (int w = 0; w < THREADS / 64; ++w) {
      if (w < wave) before += wave_sum[w];
      base += wave_sum[w];
    }
    if (e < p.E) pre[e] = before + sum - rows;
    __syncthreads();
  }
  if (tid == 0) pre[p.E] = base;
  __syncthreads();
}

struct GroupAt {
  int e, t, kg;
};
struct GroupLoads {
  u32x4 gate, up;
};

// the first expert >= e whose end lies behind `at`; there is one
template <class End>
__device__ __forceinline__ int expert_of(int e, int E, int64_t at, End end) {
  if (at < end(e)) return e;
  int last = E - 1;
  ++e;
  while (e < last) {
    const int mid = (e + last) >> 1;
    if (at < end(mid)) last = mid;
    else e = mid + 1;
  }
  return e;
}

// group c of the used rows; `e` moves forward with c
__device__ __forceinline__ GroupAt locate(const SiluQuantParams& p, const int* pre, uint32_t c, int& e) {
  const int row = (int)fastdiv(c, p.div_gpr);
  e = expert_of(e, p.E, row, [&](int i) { return pre[i + 1]; });
  return GroupAt{e, row - pre[e], (int)(c - (uint32_t)row * p.gpr)};
}
// its gate and up (16 bytes each per lane)
__device__ __forceinline__ void fetch_group(const SiluQuantParams& p, const GroupAt& g, GroupLoads& l) {
  const int lane = threadIdx.x & 15;
  const uint16_t* row = reinterpret_cast<const uint16_t*>(p.x) + ((int64_t)g.e * p.T + g.t) * 2 * p.H + (int64_t)g.kg * 128;
  l.gate = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row) + lane);
  l.up = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + p.H) + lane);
}

// T(silu(gate)) of a lane's eight gates
template <int DT, SiluTable TABLE>
__device__ __forceinline__ void look_up(const uint16_t* tbl, const uint32_t (&gate)[4], uint32_t (&silu)[8]) {
  if constexpr (TABLE == ST_NEAR) {
    u16x2 at[4], most = {0, 0};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u16x2 bits = __builtin_bit_cast(u16x2, gate[j]);
      at[j] = ((bits << (uint16_t)1) | (bits >> (uint16_t)15)) - (uint16_t)(2 * NEAR_FIRST);
      most = __builtin_elementwise_max(most, at[j]);
    }
    if (max((int)most.x, (int)most.y) < 2 * NEAR_COUNT) {
#pragma unroll
      for (int j = 0; j < 8; ++j) silu[j] = tbl[at[j >> 1][j & 1]];
      return;
    }
    tbl = g_silu_table[DT == MI355_BF16 ? 0 : 1];
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) silu[j] = tbl[(j & 1) ? (gate[j >> 1] >> 16) : (gate[j >> 1] & 0xffffu)];
}

template <int DT, SiluTable TABLE>
__device__ __forceinline__ void quant_group(const SiluQuantParams& p, const uint16_t* tbl, const GroupAt& g, const GroupLoads& cur) {
  const int lane = threadIdx.x & 15;
  const uint32_t wg[4] = {cur.gate.x, cur.gate.y, cur.gate.z, cur.gate.w};
  const uint32_t wu[4] = {cur.up.x, cur.up.y, cur.up.z, cur.up.w};
  uint32_t silu[8];
  look_up<DT, TABLE>(tbl, wg, silu);
  float v[8];
  float amax = 1e-10f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t ub = (j & 1) ? (wu[j >> 1] >> 16) : (wu[j >> 1] & 0xffffu);
    v[j] = round_to_t<DT>(mul_rn(t_bits_to_f32<DT>(silu[j]), t_bits_to_f32<DT>(ub)));  // the product of two T values is exact in fp32
    amax = fmaxf(amax, fabsf(v[j]));
  }
  amax = row16_max(amax);
  const uint32_t bits = __float_as_uint(mul_rn(amax, 1.0f / 448.0f));
  const int ex = (int)((bits >> 23) & 0xffu) - 127 + ((bits & 0x7fffffu) != 0u);  // ceil(log2(amax / 448))
  const float mul = __uint_as_float((uint32_t)(127 - ex) << 23);
  float c[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) c[j] = fminf(fmaxf(mul_rn(v[j], mul), -448.0f), 448.0f);
  int w0 = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], 0, false);
  w0 = __builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], w0, true);
  int w1 = __builtin_amdgcn_cvt_pk_fp8_f32(c[4], c[5], 0, false);
  w1 = __builtin_amdgcn_cvt_pk_fp8_f32(c[6], c[7], w1, true);
  __builtin_nontemporal_store(u32x2{(uint32_t)w0, (uint32_t)w1},
                              reinterpret_cast<u32x2*>(p.q + ((int64_t)g.e * p.T + g.t) * p.H + (int64_t)g.kg * 128 + lane * 8));
  if (lane == 0) {
    uint8_t* sb = reinterpret_cast<uint8_t*>(p.s + g.e * p.s_e + (int64_t)(g.kg >> 2) * p.s_k + g.t) + (g.kg & 3);
    *sb = (uint8_t)(ex + 127);
    if (g.kg == p.gpr - 1)  // unused bytes of the last word read as exponent 0
      for (int b = (g.kg & 3) + 1; b < 4; ++b) sb[b - (g.kg & 3)] = 0;
  }
}

template <int DT, SiluTable TABLE>
__global__ __launch_bounds__(TABLE == ST_WHOLE ? 1024 : 256) void silu_mul_quant_kernel(const SiluQuantParams p) {
  constexpr int THREADS = TABLE == ST_WHOLE ? 1024 : 256;
  constexpr int ENTRIES = TABLE == ST_WHOLE ? 65536 : TABLE == ST_NEAR ? 2 * NEAR_COUNT : 8;
  static_assert(TABLE != ST_NEAR || DT == MI355_BF16, "the near gates are bfloat16");
  __shared__ __attribute__((aligned(16))) uint16_t lds_table[ENTRIES];
  __shared__ int pre[SQ_MAX_EXPERTS + 1];
  const uint16_t* tbl = g_silu_table[DT == MI355_BF16 ? 0 : 1];
  const u32x4* entries = reinterpret_cast<const u32x4*>(tbl);
  // of the table, per thread: requested first, put into LDS last
  constexpr int NEAR_PIECES = NEAR_COUNT / 8, NEAR_EACH = (NEAR_PIECES + THREADS - 1) / THREADS;
  constexpr int PIECES = TABLE == ST_WHOLE ? 65536 / 8 / THREADS : TABLE == ST_NEAR ? 2 * NEAR_EACH : 1;
  u32x4 piece[PIECES];
  if constexpr (TABLE == ST_WHOLE) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) piece[i] = entries[i * THREADS + threadIdx.x];
  } else if constexpr (TABLE == ST_NEAR) {
#pragma unroll
    for (int i = 0; i < NEAR_EACH; ++i) {
      const int at = NEAR_FIRST / 8 + min(i * THREADS + (int)threadIdx.x, NEAR_PIECES - 1);
      piece[2 * i] = entries[at], piece[2 * i + 1] = entries[0x8000 / 8 + at];
    }
  }
  scan_rows<THREADS>(p, pre);
  const uint32_t groups = (uint32_t)pre[p.E] * p.gpr;
  const uint32_t stride = gridDim.x * (THREADS / 16);
  uint32_t c = blockIdx.x * (THREADS / 16) + (threadIdx.x >> 4);
  int e = 0;
  GroupAt at{0, 0, 0}, at1{0, 0, 0}, at2{0, 0, 0};
  GroupLoads cur, nxt, nxt2;
  if (c < groups) at = locate(p, pre, c, e), fetch_group(p, at, cur);
  if constexpr (TABLE == ST_WHOLE) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) reinterpret_cast<u32x4*>(lds_table)[i * THREADS + threadIdx.x] = piece[i];
  } else if constexpr (TABLE == ST_NEAR) {
#pragma unroll
    for (int i = 0; i < NEAR_EACH; ++i) {
      u32x4* to = reinterpret_cast<u32x4*>(lds_table) + 2 * min(i * THREADS + (int)threadIdx.x, NEAR_PIECES - 1);
      const u32x4 pos = piece[2 * i], neg = piece[2 * i + 1];
      const u32x4 even = (pos & 0xffffu) | (neg << 16), odd = (pos >> 16) | (neg & 0xffff0000u);
      to[0] = u32x4{even.x, odd.x, even.y, odd.y}, to[1] = u32x4{even.z, odd.z, even.w, odd.w};
    }
  }
  if constexpr (TABLE != ST_IN_PLACE) {
    __syncthreads();
    tbl = lds_table;
  }
  if (c + stride < groups) at1 = locate(p, pre, c + stride, e), fetch_group(p, at1, nxt);  // (groups < 2^30: no overflow)
  for (; c < groups; c += stride) {
    // two groups ahead: three 32-byte requests per lane in flight
    if (c + 2 * stride < groups) at2 = locate(p, pre, c + 2 * stride, e), fetch_group(p, at2, nxt2);
    quant_group<DT, TABLE>(p, tbl, at, cur);
    cur = nxt, nxt = nxt2;
    at = at1, at1 = at2;
  }
  if (!p.zero_rest) return;
  // the unused rows, a wave per row: dead row d of the launch is row pre[e + 1] - pre[e] + (d - (e T - pre[e])) of expert e
  const int lane = threadIdx.x & 63;
  const int64_t dead = (int64_t)p.E * p.T - pre[p.E];
  int ez = 0;
  for (int64_t d = (int64_t)blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6); d < dead; d += (int64_t)gridDim.x * (THREADS / 64)) {
    ez = expert_of(ez, p.E, d, [&](int i) { return (int64_t)(i + 1) * p.T - pre[i + 1]; });
    const int64_t t = pre[ez + 1] - pre[ez] + (d - ((int64_t)ez * p.T - pre[ez]));
    uint8_t* row = p.q + ((int64_t)ez * p.T + t) * p.H;
    for (int64_t i = lane * 8; i < p.H; i += 64 * 8) __builtin_nontemporal_store(u32x2{0u, 0u}, reinterpret_cast<u32x2*>(row + i));
    for (int w = lane; w < (p.gpr + 3) / 4; w += 64) p.s[ez * p.s_e + (int64_t)w * p.s_k + t] = 0u;
  }
}

int silu_mul_group_quant(const char* what, const void* x, int x_dtype, void* q, void* s_words, int64_t E, int64_t T, int64_t H,
                         const int32_t* masked_m, int64_t s_expert_stride, int64_t s_k_stride, bool zero_rest, void* stream) {
  clear_error();
  MI355_REQUIRE(E >= 0 && T >= 0 && H >= 0, MI355_ERR_INVALID_ARGUMENT, "%s: negative shape", what);
  MI355_REQUIRE(x_dtype == MI355_F16 || x_dtype == MI355_BF16, MI355_ERR_INVALID_ARGUMENT,
                "%s: input must be float16 or bfloat16", what);
  if (E == 0 || T == 0 || H == 0) return MI355_OK;
  MI355_REQUIRE(x && q && s_words, MI355_ERR_INVALID_ARGUMENT, "%s: null pointer", what);
  MI355_REQUIRE(H % 128 == 0, MI355_ERR_UNSUPPORTED, "%s: the hidden size must be a multiple of the group size 128", what);
  MI355_REQUIRE(((uintptr_t)x % 16 == 0) && ((uintptr_t)q % 8 == 0) && ((uintptr_t)s_words % 4 == 0), MI355_ERR_INVALID_ARGUMENT,
                "%s: input must be 16-byte, output 8-byte and scales 4-byte aligned", what);
  const int64_t gpr = H / 128;
  MI355_REQUIRE(E * T < (1ll << 31) && H < (1ll << 31), MI355_ERR_INVALID_ARGUMENT, "%s: shape out of range", what);
  hipStream_t st = static_cast<hipStream_t>(stream);
  for (int64_t e0 = 0; e0 < E; e0 += SQ_MAX_EXPERTS) {
    SiluQuantParams p;
    p.E = (int)(E - e0 < SQ_MAX_EXPERTS ? E - e0 : SQ_MAX_EXPERTS);
    p.T = T, p.H = H, p.gpr = (int)gpr, p.div_gpr = make_fastdiv((uint32_t)gpr);
    p.x = static_cast<const uint16_t*>(x) + e0 * T * 2 * H;
    p.q = static_cast<uint8_t*>(q) + e0 * T * H;
    p.s = static_cast<uint32_t*>(s_words) + e0 * s_expert_stride;
    p.masked_m = masked_m ? masked_m + e0 : nullptr;
    p.s_e = s_expert_stride, p.s_k = s_k_stride;
    p.zero_rest = zero_rest;
    const int64_t groups = p.E * T * gpr;
    MI355_REQUIRE(groups < (1ll << 30), MI355_ERR_INVALID_ARGUMENT, "%s: too many groups", what);
    const bool bf16 = x_dtype == MI355_BF16;
    if (bf16 && groups <= (masked_m ? SQ_NEAR_GROUPS_MASKED : SQ_NEAR_GROUPS)) {
      const dim3 grid((unsigned)std::min<int64_t>((groups + 15) / 16, SQ_NEAR_WORKGROUPS));
      launch_kernel((silu_mul_quant_kernel<MI355_BF16, ST_NEAR>), grid, dim3(256), 0, st, p);
    } else if (bf16) {
      launch_kernel((silu_mul_quant_kernel<MI355_BF16, ST_WHOLE>), dim3(256), dim3(1024), 0, st, p);
    } else if (groups <= (masked_m ? SQ_IN_PLACE_GROUPS_MASKED : SQ_IN_PLACE_GROUPS)) {
      launch_kernel((silu_mul_quant_kernel<MI355_F16, ST_IN_PLACE>), dim3((unsigned)((groups + 15) / 16)), dim3(256), 0, st, p);
    } else {
      launch_kernel((silu_mul_quant_kernel<MI355_F16, ST_WHOLE>), dim3(256), dim3(1024), 0, st, p);
    }
    const int rc = check_launch(what);
    if (rc != MI355_OK) return rc;
  }
  return MI355_OK;
}

}  // namespace
}  // namespace mi355

using namespace mi355;

extern "C" int mi355_silu_mul_group_quant_fp8(const void* x, int x_dtype, void* q, void* s_words, int64_t E, int64_t T,
                                              int64_t H, const int32_t* masked_m, int64_t s_expert_stride,
                                              int64_t s_k_stride, void* stream) {
  return silu_mul_group_quant("mi355_silu_mul_group_quant_fp8", x, x_dtype, q, s_words, E, T, H, masked_m, s_expert_stride, s_k_stride,
                              false, stream);
}

extern "C" int mi355_silu_mul_group_quant_fp8_zero_rest(const void* x, int x_dtype, void* q, void* s_words, int64_t E, int64_t T,
                                                        int64_t H, const int32_t* masked_m, int64_t s_expert_stride,
                                                        int64_t s_k_stride, void* stream) {
  return silu_mul_group_quant("mi355_silu_mul_group_quant_fp8_zero_rest", x, x_dtype, q, s_words, E, T, H, masked_m, s_expert_stride,
                              s_k_stride, true, stream);
}
