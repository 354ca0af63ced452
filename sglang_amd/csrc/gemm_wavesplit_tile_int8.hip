// Small-tile INT8 GEMM with K split over the waves (gemm_wavesplit_tile.h): exact int32 sums.
#include "gemm_wavesplit_tile.h"

namespace mi355 {
int launch_int8_wavesplit_tile(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_of<AR_INT8>(p, bm, bn, stream, what);
}
int launch_int8_wavesplit_tile_quant(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_wavesplit_tile_quant<AR_INT8, TQ_ROW>(p, bm, bn, stream, what);
}
}  // namespace mi355
