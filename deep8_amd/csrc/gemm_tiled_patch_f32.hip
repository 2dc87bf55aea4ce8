// Tiled GEMM, fp32: products with a patch-matrix operand (gemm_tiled_launch.h).
#include "gemm_tiled_launch.h"

namespace d8 {

int gemm_tiled_patch_f32(const GemmArgs &g, int transB, hipStream_t stream) { return launch_patch<float>(g, transB, stream); }

}  // namespace d8
