// Small-tile FP8 GEMM with K split over the waves (gemm_wavesplit_tile.h): one scale per token and channel.
#include "gemm_wavesplit_tile.h"

namespace mi355 {
int launch_fp8_wavesplit_tile_unit(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_of<AR_UNIT>(p, bm, bn, stream, what);
}
int launch_fp8_wavesplit_tile_unit_quant(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_quant<AR_UNIT, TQ_ROW>(p, bm, bn, stream, what);
}
}  // namespace mi355
