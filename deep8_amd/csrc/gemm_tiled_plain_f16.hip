// Tiled GEMM, fp16: products of real matrices (gemm_tiled_launch.h).
#include "gemm_tiled_launch.h"

namespace d8 {

int gemm_tiled_plain_f16(const GemmArgs &g, int transA, int transB, hipStream_t stream) { return launch_plain<f16>(g, transA, transB, stream); }

}  // namespace d8
