// Both gradients of a convolution in half as one launch (gemm_tiled_pair_kernel, gemm_tiled_kernel.h), where K may cut gx's last
// step short and either may be split along its reduction (the caller reduces).
#include "gemm_tiled_kernel.h"

namespace d8 {

static bool pair_tiles(const GemmArgs &gx, const GemmArgs &gy, TileId &tx, TileId &ty) {
    if (gx.virt != VIRT_A_ROWS || gy.virt != VIRT_B_KROWS || gx.batch != 1 || gy.batch != 1 || gx.tail_splits || gy.tail_splits) return false;
    tx = choose_tile<f16, true, false, VIRT_A_ROWS>(gx), ty = choose_tile<f16, false, false, VIRT_B_KROWS>(gy);
    return (tx == TILE_64x64 || tx == TILE_64x128 || tx == TILE_128x128 || tx == TILE_128x64) && (ty == TILE_128x128 || ty == TILE_64x128 || ty == TILE_64x64);
}

bool gemm_tiled_rows_pair_tiles(const GemmArgs &gx, const GemmArgs &gy) {
    TileId tx, ty;
    if (!pair_tiles(gx, gy, tx, ty)) return false;
    int mx, nx, my, ny;
    grid_of(tx, gx, mx, nx);
    grid_of(ty, gy, my, ny);
    return (long)mx * nx * gx.splits + (long)my * ny * gy.splits < 0x7fffffffL;
}

template <typename X>
static int launch_y(TileId ty, const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    switch (ty) {
        case TILE_128x128: return launch_pair_tiles<X, typename TileOf<f16, 128, 128, false, false, VIRT_B_KROWS>::type, EDGE_PIECES>(gx, gy, stream);
        case TILE_64x128: return launch_pair_tiles<X, typename TileOf<f16, 64, 128, false, false, VIRT_B_KROWS>::type, EDGE_PIECES>(gx, gy, stream);
        default: return launch_pair_tiles<X, typename TileOf<f16, 64, 64, false, false, VIRT_B_KROWS>::type, EDGE_PIECES>(gx, gy, stream);
    }
}

int gemm_tiled_rows_pair_launch(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    TileId tx, ty;
    if (!pair_tiles(gx, gy, tx, ty)) return fail(D8_ERR_ARGUMENT, "gemm_tiled_rows_pair_launch: no kernel for this pair of tiles");
    switch (tx) {
        case TILE_64x64: return launch_y<typename TileOf<f16, 64, 64, true, false, VIRT_A_ROWS>::type>(ty, gx, gy, stream);
        case TILE_64x128: return launch_y<typename TileOf<f16, 64, 128, true, false, VIRT_A_ROWS>::type>(ty, gx, gy, stream);
        case TILE_128x128: return launch_y<typename TileOf<f16, 128, 128, true, false, VIRT_A_ROWS>::type>(ty, gx, gy, stream);
        default: return launch_y<typename TileOf<f16, 128, 64, true, false, VIRT_A_ROWS>::type>(ty, gx, gy, stream);
    }
}

}  // namespace d8
