// Both gradients of a convolution as one launch, fp32: x's product over classes of output pixels (gemm_tiled_pair_kept.h).
#include "gemm_tiled_pair_kept.h"

namespace d8 {

int gemm_tiled_pair_classes_f32(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) { return kept_launch<float, VIRT_A_CLASSES>(gx, gy, stream); }

}  // namespace d8
