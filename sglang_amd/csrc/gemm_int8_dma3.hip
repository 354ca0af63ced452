// Mid-M per-token x per-channel INT8 GEMM for gfx950: the tile of gemm_dma_tile.h with v_mfma_i32_16x16x64_i8, two per 16 x 16
// tile and 128-byte K block (chunk q of both operands' rows, then chunk q + 4), exact int32 accumulation.  Tiling and split as
// for FP8 (dma3_plan); the 128-channel tiles fill the chip for layers with few channels.  Optional split along K: int32
// partials to the workspace, the ordered reduce applies the epilogue.
#include "gemm_dma_tile.h"

namespace mi355 {

int launch_int8_dma3(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_dma_tile_of<AR_INT8>(p, bm, bn, stream, what);
}

}  // namespace mi355
