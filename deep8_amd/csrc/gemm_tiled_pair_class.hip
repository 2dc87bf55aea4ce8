// Both gradients of a strided Conv2d in half as one launch (gemm_tiled_pair_kernel, gemm_tiled_kernel.h): gx runs over the
// classes of output pixels (NN), gy has patch k-rows as B (TN) and may be split along its reduction (the caller reduces).
#include "gemm_tiled_kernel.h"

namespace d8 {

bool gemm_tiled_class_pair_tiles(const GemmArgs &gx, const GemmArgs &gy) {
    if (gx.virt != VIRT_A_CLASSES || gy.virt != VIRT_B_KROWS || gx.splits != 1 || gx.batch != 1 || gy.batch != 1 || gy.tail_splits || gy.tile_hint) return false;
    const TileId ty = choose_tile<f16, false, false, VIRT_B_KROWS>(gy);
    if (ty != TILE_128x128 && ty != TILE_64x128 && ty != TILE_64x64) return false;
    int my, ny;
    grid_of(ty, gy, my, ny);
    return (long)ceil_div(gx.M, 128) * ceil_div(gx.N, gx.N < 128 ? 64 : 128) * gx.ncls + (long)my * ny * gy.splits < 0x7fffffffL;
}

template <typename X, int EDGE>
static int launch_y(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    switch (choose_tile<f16, false, false, VIRT_B_KROWS>(gy)) {
        case TILE_128x128: return launch_pair_tiles<X, typename TileOf<f16, 128, 128, false, false, VIRT_B_KROWS>::type, EDGE>(gx, gy, stream);
        case TILE_64x128: return launch_pair_tiles<X, typename TileOf<f16, 64, 128, false, false, VIRT_B_KROWS>::type, EDGE>(gx, gy, stream);
        default: return launch_pair_tiles<X, typename TileOf<f16, 64, 64, false, false, VIRT_B_KROWS>::type, EDGE>(gx, gy, stream);
    }
}

// (the tiles of gemm_tiled_launch.h; a last K step that K cuts short asks nothing of the filter gradient, whose rows end with
// their buffer)
int gemm_tiled_class_pair_launch(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    if (!gemm_tiled_class_pair_tiles(gx, gy)) return fail(D8_ERR_ARGUMENT, "gemm_tiled_class_pair_launch: no kernel for this pair of tiles");
    typedef typename TileOf<f16, 128, 64, true, false, VIRT_A_CLASSES>::type Narrow;
    typedef typename TileOf<f16, 128, 128, true, false, VIRT_A_CLASSES>::type Wide;
    if (gx.K % 64) return gx.N < 128 ? launch_y<Narrow, EDGE_PIECES>(gx, gy, stream) : launch_y<Wide, EDGE_PIECES>(gx, gy, stream);
    return gx.N < 128 ? launch_y<Narrow, EDGE_NONE>(gx, gy, stream) : launch_y<Wide, EDGE_NONE>(gx, gy, stream);
}

}  // namespace d8
