// GEMM of short K with the weight in registers (gemm_resident.h): scales in the epilogue.
#include "gemm_resident.h"

namespace mi355 {
int launch_fp8_resident_unit(GemmParams& p, int ranges, hipStream_t stream, const char* what) { return launch_resident_of<AR_UNIT>(p, ranges, stream, what); }
}  // namespace mi355
