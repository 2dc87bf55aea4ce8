// The two gradients of a mid-size MatrixMultiply in one launch (gemm_tiled_pair_plain.h), fp32, where K cuts a last step of either short.
#include "gemm_tiled_pair_plain.h"

namespace d8 {

int gemm_tiled_plain_pair_pieces_f32(const GemmArgs &g0, const GemmArgs &g1, hipStream_t stream) { return launch_plain_pair<float, EDGE_PIECES>(g0, g1, stream); }

}  // namespace d8
