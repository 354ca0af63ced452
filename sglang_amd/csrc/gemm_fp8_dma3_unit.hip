// Mid-M FP8 GEMM with one scale per token and channel (fp8_scaled_mm): no scales in the K loop, both applied in the epilogue, or
// by the ordered reduce after a K split (see gemm_dma_tile.h).  K = 4096 -> N = 28672 at 160 tokens took 56 us when the token
// scale rode along as a block scale: a relayout launch first, and a promotion FMA per product that nothing needed.
#include "gemm_dma_tile.h"

namespace mi355 {

int launch_fp8_dma3_unit(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_dma_tile_of<AR_UNIT>(p, bm, bn, stream, what);
}

}  // namespace mi355
