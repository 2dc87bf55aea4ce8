// Both gradients of a convolution as one launch, fp32: x's product on patch rows (gemm_tiled_pair_kept.h).
#include "gemm_tiled_pair_kept.h"

namespace d8 {

SharedLaunch gemm_tiled_kept_pair_tiles_f32(const GemmArgs &gx, const GemmArgs &gy) {
    TileId tx, ty;
    return kept_tiles<float>(gx, gy, tx, ty);
}

int gemm_tiled_pair_rows_f32(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) { return kept_launch<float, VIRT_A_ROWS>(gx, gy, stream); }

}  // namespace d8
