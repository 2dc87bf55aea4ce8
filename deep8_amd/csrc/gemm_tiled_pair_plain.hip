// The two gradients of a mid-size MatrixMultiply in one launch (gemm_tiled_pair_plain.h): whole K steps, and copies of odd operands.
#include "gemm_tiled_pair_plain.h"

namespace d8 {

long gemm_tiled_plain_pair_workgroups(int dtype, const GemmArgs &g0, const GemmArgs &g1) {
    TileId t0, t1;
    if (g0.virt != VIRT_NONE || g1.virt != VIRT_NONE || g0.tail_splits || g1.tail_splits) return 0;
    if (!(dtype == D8_FLOAT16 ? plain_pair_tiles<f16>(g0, g1, t0, t1) : plain_pair_tiles<float>(g0, g1, t0, t1))) return 0;
    int m0, n0, m1, n1;
    grid_of(t0, g0, m0, n0);
    grid_of(t1, g1, m1, n1);
    const long wg0 = (long)m0 * n0 * g0.batch * g0.splits, wg1 = (long)m1 * n1 * g1.batch * g1.splits;
    if (wg0 + wg1 <= 2L * cu_count() || g0.packed) return wg0 + wg1;
    const bool tail = dtype == D8_FLOAT32 ? leaves_a_tail(g0, t0, wg0, g1, t1, wg1) : leaves_a_half_tail(g0, t0, wg0, g1, t1, wg1);
    return tail ? 0 : wg0 + wg1;
}

int gemm_tiled_plain_pair_launch(int dtype, const GemmArgs &g0, const GemmArgs &g1, hipStream_t stream) {
    const bool half = dtype == D8_FLOAT16;
    if (half && g0.packed) return launch_plain_pair<f16, EDGE_ANY>(g0, g1, stream);
    const int BK = half ? 64 : 32;
    if (g0.K % BK || g1.K % BK) return half ? gemm_tiled_plain_pair_pieces_f16(g0, g1, stream) : gemm_tiled_plain_pair_pieces_f32(g0, g1, stream);
    return half ? launch_plain_pair<f16, EDGE_NONE>(g0, g1, stream) : launch_plain_pair<float, EDGE_NONE>(g0, g1, stream);
}

}  // namespace d8
