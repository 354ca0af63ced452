// GEMM of short K with the weight in registers (gemm_resident.h): packed exponents.
#include "gemm_resident.h"

namespace mi355 {
int launch_fp8_resident_ue8m0(GemmParams& p, int ranges, hipStream_t stream, const char* what) { return launch_resident_of<AR_UE8M0>(p, ranges, stream, what); }
}  // namespace mi355
