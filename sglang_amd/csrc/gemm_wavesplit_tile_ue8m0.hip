// Small-tile FP8 GEMM with K split over the waves (gemm_wavesplit_tile.h): packed exponents applied by the MFMA.
#include "gemm_wavesplit_tile.h"

namespace mi355 {
int launch_fp8_wavesplit_tile_ue8m0(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_of<AR_UE8M0>(p, bm, bn, stream, what);
}
int launch_fp8_wavesplit_tile_ue8m0_quant(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_quant<AR_UE8M0, TQ_GROUP>(p, bm, bn, stream, what);
}
}  // namespace mi355
