// GEMM of short K with the weight in registers (gemm_resident.h): INT8.
#include "gemm_resident.h"

namespace mi355 {
int launch_int8_resident(GemmParams& p, int ranges, hipStream_t stream, const char* what) { return launch_resident_of<AR_INT8>(p, ranges, stream, what); }
}  // namespace mi355
