// Mid-M FP8 GEMM with packed power-of-two (UE8M0) scales on both operands, applied by the MFMA (see gemm_dma_tile.h).
#include "gemm_dma_tile.h"

namespace mi355 {

int launch_fp8_dma3_ue8m0(GemmParams& p, int bm, int bn, hipStream_t stream, const char* what) {
  return launch_dma_tile_of<AR_UE8M0>(p, bm, bn, stream, what);
}

}  // namespace mi355
