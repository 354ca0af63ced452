// Shared host/device helpers of the gfx950 quantized-linear kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <cstdarg>
#include <cstdio>
#include <tuple>

#include "mi355_qlinear.h"

namespace mi355 {

// ---- error reporting (host) -------------------------------------------------------------
void set_error(const char* fmt, ...);  // defined in error.cpp; stores a thread-local message
void clear_error();

#define MI355_REQUIRE(cond, code, ...) \
  do {                                 \
    if (!(cond)) {                     \
      ::mi355::set_error(__VA_ARGS__); \
      return (code);                   \
    }                                  \
  } while (0)

// kernel<<<grid, block, lds, stream>>>(args...) as one call of the runtime: the launch syntax makes three of it, the configuration on to and off a
// per-thread stack among them.  A linear, a quantizer and the grouped GEMM of a few rows are bound by these calls; host us of one call of the
// Python function, <<<>>> / this: one launch block FP8 5.2 / 4.45, INT8 5.0 / 4.3, group quantizer 5.8 to 6.2 / 5.2 to 5.5; two launches
// block FP8 8.75 / 6.95, INT8 8.45 / 6.9, grouped 9.05 / 7.6.  Errors are the runtime's last error, as behind <<<>>> (check_launch).
template <class... Params, class... Args>
inline void launch_kernel(void (*kernel)(Params...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, const Args&... args) {
  static_assert(sizeof...(Params) == sizeof...(Args), "an argument per parameter");
  std::tuple<Params...> held(args...);
  std::apply([&](Params&... p) {
    void* pointers[] = {&p...};
    (void)hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, pointers, lds, stream);
  }, held);
}
inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return MI355_ERR_LAUNCH;
  }
  return MI355_OK;
}

inline size_t dtype_size(int dt) {
  switch (dt) {
    case MI355_F32: return 4;
    case MI355_I32: return 4;
    case MI355_F16: return 2;
    case MI355_BF16: return 2;
    default: return 1;
  }
}

// Division of a 31-bit unsigned numerator by a run-time constant with one multiply-high and a shift.
struct FastDiv {
  uint32_t mul, shift, div;
};
inline FastDiv make_fastdiv(uint32_t d) {
  // ceil(2^(32+s) / d) with s = ceil(log2 d); exact for numerators below 2^31.
  FastDiv f;
  f.div = d;
  uint32_t s = 0;
  while ((1ull << s) < d) ++s;
  f.shift = s;
  f.mul = (uint32_t)((((1ull << 32) * ((1ull << s) - d)) / d) + 1);
  return f;
}

// ---- device helpers ---------------------------------------------------------------------
__device__ __forceinline__ uint32_t fastdiv(uint32_t n, const FastDiv& f) {
  uint32_t t = __umulhi(n, f.mul);
  return (t + n) >> f.shift;  // n < 2^31, so t + n cannot overflow
}

// Separately rounded fp32 multiply and add: the INT8 epilogue contract is mul, mul, add, and no code motion may fuse two of them into an FMA (a fused
// result differs in the last bit of the 16-bit output about once in 10^5 elements), nor one of them into a conversion (v_fma_mixlo_f16 rounds a product to
// fp16 once).  So the result passes through an empty asm, and the pragma takes the leave to fuse off the operation itself, which -ffp-contract=fast would
// pass over.  The operation is not asm: the compiler does not see what asm reads, and would not wait for an MFMA's result in front of it.
__device__ __forceinline__ float mul_rn(float a, float b) {
#pragma clang fp contract(off)
  float r = a * b;
  asm("" : "+v"(r));
  return r;
}
__device__ __forceinline__ float add_rn(float a, float b) {
#pragma clang fp contract(off)
  float r = a + b;
  asm("" : "+v"(r));
  return r;
}

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t h) { return __uint_as_float(h << 16); }

// Two fp32 values to packed bf16 / fp16 (lo in bits 0..15), round to nearest even, NaN stays NaN: one instruction of gfx950 each.  As the
// compiler's own conversions and not as asm: it does not see what asm reads, so it would not wait for an MFMA's result in front of it.
template <class T16>
__device__ __forceinline__ uint32_t pack_16x2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef T16 t16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), t16x2));
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) { return pack_16x2<__bf16>(lo, hi); }
__device__ __forceinline__ uint32_t pack_f16x2(float lo, float hi) { return pack_16x2<_Float16>(lo, hi); }
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) { return pack_bf16x2(f, f) & 0xffffu; }

__device__ __forceinline__ uint32_t f32_to_f16_bits(float f) {
  return (uint32_t)__half_as_ushort(__float2half_rn(f));
}

__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
  return __half2float(__ushort_as_half((unsigned short)h));
}

}  // namespace mi355
