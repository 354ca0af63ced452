// Small-tile FP8 GEMM with K split over the waves (gemm_wavesplit_tile.h): fp32 block scales.
#include "gemm_wavesplit_tile.h"

namespace mi355 {
int launch_fp8_wavesplit_tile(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_of<AR_F32>(p, bm, bn, stream, what);
}
int launch_fp8_wavesplit_tile_quant(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_quant<AR_F32, TQ_GROUP>(p, bm, bn, stream, what);
}
}  // namespace mi355
