// GEMM of short K with the weight in registers (gemm_resident.h): fp32 block scales.
#include "gemm_resident.h"

namespace mi355 {
int launch_fp8_resident(GemmParams& p, int ranges, hipStream_t stream, const char* what) { return launch_resident_of<AR_F32>(p, ranges, stream, what); }
}  // namespace mi355
