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
// run time.  Two forms, chosen by the number of groups (SQ_SMALL_GROUPS):
//   * many: 256 workgroups of 1024 threads (one per CU), each with its table copied into LDS (128 of the CU's 160 KB);
//   * few: the copy alone would take longer than the work: 256-thread workgroups that look up in the table where it lies.
// A 16-lane row of a wave takes a group (8 values per lane: one 16-byte load of gate, one of up, eight lookups, one 8-byte
// store), the loads of the next two groups are requested before the current one is processed.  4 B in and 1 B out per value.
//
// Rows in use are dealt out over the whole launch: every workgroup scans the experts' row counts (they are on the device) and
// walks the list of used rows of all experts with the grid's stride.  With a fixed share of the workgroups per expert the
// fullest expert set the time: 32 experts of 256 rows, half of them used on average, took 17.8 us, the fills 5.5 + 1.8 more.
#include "common.h"

namespace mi355 {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __attribute__((aligned(16))) const uint16_t g_silu_table[2][65536] = {
#include "silu_table.inc"
};

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
// Up to here the looked-up table stays where it lies.  Measured, us a call, in place / in LDS: 24000 groups 6.8 / 8.3, 65536
// 13.3 / 11.0; masked with about half of the rows in use 32768 7.1 / 10.3, 65536 9.9 / 12.9, 131072 17.8 / 15.6, 262144 30.6 / 23.4.
constexpr int64_t SQ_SMALL_GROUPS = 49152, SQ_SMALL_GROUPS_MASKED = 98304;

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

// group c of the used rows; `e` walks forward with c
__device__ __forceinline__ GroupAt locate(const SiluQuantParams& p, const int* pre, uint32_t c, int& e) {
  const int row = (int)fastdiv(c, p.div_gpr);
  while (row >= pre[e + 1]) ++e;
  return GroupAt{e, row - pre[e], (int)(c - (uint32_t)row * p.gpr)};
}
// its gate and up (16 bytes each per lane)
__device__ __forceinline__ void fetch_group(const SiluQuantParams& p, const GroupAt& g, GroupLoads& l) {
  const int lane = threadIdx.x & 15;
  const uint16_t* row = reinterpret_cast<const uint16_t*>(p.x) + ((int64_t)g.e * p.T + g.t) * 2 * p.H + (int64_t)g.kg * 128;
  l.gate = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row) + lane);
  l.up = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + p.H) + lane);
}

template <int DT>
__device__ __forceinline__ void quant_group(const SiluQuantParams& p, const uint16_t* tbl, const GroupAt& g, const GroupLoads& cur) {
  const int lane = threadIdx.x & 15;
  const uint32_t wg[4] = {cur.gate.x, cur.gate.y, cur.gate.z, cur.gate.w};
  const uint32_t wu[4] = {cur.up.x, cur.up.y, cur.up.z, cur.up.w};
  float v[8];
  float amax = 1e-10f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t gb = (j & 1) ? (wg[j >> 1] >> 16) : (wg[j >> 1] & 0xffffu);
    const uint32_t ub = (j & 1) ? (wu[j >> 1] >> 16) : (wu[j >> 1] & 0xffffu);
    const float sl = t_bits_to_f32<DT>(tbl[gb]);                    // T(silu(gate))
    v[j] = round_to_t<DT>(mul_rn(sl, t_bits_to_f32<DT>(ub)));       // the product of two T values is exact in fp32
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

template <int DT, bool LDS_TABLE>
__global__ __launch_bounds__(LDS_TABLE ? 1024 : 256) void silu_mul_quant_kernel(const SiluQuantParams p) {
  constexpr int THREADS = LDS_TABLE ? 1024 : 256;
  __shared__ __attribute__((aligned(16))) uint16_t lds_table[LDS_TABLE ? 65536 : 1];
  __shared__ int pre[SQ_MAX_EXPERTS + 1];
  const uint16_t* tbl = g_silu_table[DT == MI355_BF16 ? 0 : 1];
  constexpr int PIECES = 65536 * 2 / 16 / 1024;  // of the table, per thread: requested first, put into LDS last
  u32x4 piece[LDS_TABLE ? PIECES : 1];
  if constexpr (LDS_TABLE) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) piece[i] = reinterpret_cast<const u32x4*>(tbl)[i * THREADS + threadIdx.x];
  }
  scan_rows<THREADS>(p, pre);
  const uint32_t groups = (uint32_t)pre[p.E] * p.gpr;
  const uint32_t stride = gridDim.x * (THREADS / 16);
  uint32_t c = blockIdx.x * (THREADS / 16) + (threadIdx.x >> 4);
  int e = 0;
  GroupAt at{0, 0, 0}, at1{0, 0, 0}, at2{0, 0, 0};
  GroupLoads cur, nxt, nxt2;
  if (c < groups) at = locate(p, pre, c, e), fetch_group(p, at, cur);
  if constexpr (LDS_TABLE) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) reinterpret_cast<u32x4*>(lds_table)[i * THREADS + threadIdx.x] = piece[i];
    __syncthreads();
    tbl = lds_table;
  }
  if (c + stride < groups) at1 = locate(p, pre, c + stride, e), fetch_group(p, at1, nxt);  // (groups < 2^30: no overflow)
  for (; c < groups; c += stride) {
    // two groups ahead: three 32-byte requests per lane in flight
    if (c + 2 * stride < groups) at2 = locate(p, pre, c + 2 * stride, e), fetch_group(p, at2, nxt2);
    quant_group<DT>(p, tbl, at, cur);
    cur = nxt, nxt = nxt2;
    at = at1, at1 = at2;
  }
  if (!p.zero_rest) return;
  // the unused rows, a wave per row: dead row d of the launch is row pre[e + 1] - pre[e] + (d - (e T - pre[e])) of expert e
  const int lane = threadIdx.x & 63;
  const int64_t dead = (int64_t)p.E * p.T - pre[p.E];
  int ez = 0;
  for (int64_t d = (int64_t)blockIdx.x * (THREADS / 64) + (threadIdx.x >> 6); d < dead; d += (int64_t)gridDim.x * (THREADS / 64)) {
    while (d >= (int64_t)(ez + 1) * p.T - pre[ez + 1]) ++ez;
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
    if (groups <= (masked_m ? SQ_SMALL_GROUPS_MASKED : SQ_SMALL_GROUPS)) {
      const dim3 grid((unsigned)((groups + 15) / 16));
      if (x_dtype == MI355_BF16) hipLaunchKernelGGL((silu_mul_quant_kernel<MI355_BF16, false>), grid, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((silu_mul_quant_kernel<MI355_F16, false>), grid, dim3(256), 0, st, p);
    } else {
      if (x_dtype == MI355_BF16) hipLaunchKernelGGL((silu_mul_quant_kernel<MI355_BF16, true>), dim3(256), dim3(1024), 0, st, p);
      else hipLaunchKernelGGL((silu_mul_quant_kernel<MI355_F16, true>), dim3(256), dim3(1024), 0, st, p);
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
