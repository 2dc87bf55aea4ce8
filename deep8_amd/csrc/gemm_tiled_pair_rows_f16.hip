// Both gradients of a convolution as one launch, half: x's product on patch rows (gemm_tiled_pair_kept.h).
#include "gemm_tiled_pair_kept.h"

namespace d8 {

SharedLaunch gemm_tiled_kept_pair_tiles_f16(const GemmArgs &gx, const GemmArgs &gy) {
    TileId tx, ty;
    return kept_tiles<f16>(gx, gy, tx, ty);
}

int gemm_tiled_pair_rows_f16(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) { return kept_launch<f16, VIRT_A_ROWS>(gx, gy, stream); }

}  // namespace d8
