// Both gradients of a convolution as one launch (gemm_tiled_pair_kernel, gemm_tiled_kernel.h), each tiled and cut as it would be
// alone: K may cut gx's last step short and either may be split along its reduction (the caller reduces).  gx has patch rows as A
// or runs over the classes of output pixels.  Included by the translation units that instantiate it, one per element type.
#ifndef DEEP8_AMD_GEMM_TILED_PAIR_KEPT_H
#define DEEP8_AMD_GEMM_TILED_PAIR_KEPT_H

#include "gemm_tiled_kernel.h"

namespace d8 {

template <typename E>
static bool kept_tiles(const GemmArgs &gx, const GemmArgs &gy, TileId &tx, TileId &ty) {
    if (gy.virt != VIRT_B_KROWS || gx.batch != 1 || gy.batch != 1 || gx.tail_splits || gy.tail_splits) return false;
    if (gx.virt == VIRT_A_CLASSES) {  // (the tiles of gemm_tiled_launch.h)
        if (gx.splits != 1) return false;
        tx = sizeof(E) == 4 && gx.N <= 32 ? TILE_128x32 : gx.N < 128 ? TILE_128x64 : TILE_128x128;
    } else if (gx.virt == VIRT_A_ROWS) {
        tx = choose_tile<E, true, false, VIRT_A_ROWS>(gx);
    } else {
        return false;
    }
    ty = choose_tile<E, false, false, VIRT_B_KROWS>(gy);
    const bool x_ok = tx == TILE_64x64 || tx == TILE_64x128 || tx == TILE_128x128 || tx == TILE_128x64 || (sizeof(E) == 4 && tx == TILE_128x32);
    if (!x_ok || (ty != TILE_128x128 && ty != TILE_64x128 && ty != TILE_64x64)) return false;
    // (fp32 on 128 x 128 tiles in both: bound by the matrix pipe either way, and side by side they miss the caches more often.
    // DeConv2d 59 x 7x7x256 -> 240 4x4 stride 2 124.4 us apart, 135.9 in one launch)
    if (sizeof(E) == 4 && gx.virt == VIRT_A_ROWS && tx == TILE_128x128 && ty == TILE_128x128) return false;
    int mx, nx, my, ny;
    grid_of(ty, gy, my, ny);
    if (sizeof(E) == 4 && gx.virt == VIRT_A_ROWS) {
        // (fp32: all workgroups at once, two to a compute unit.  With more a smaller tile's product, of which three would fit,
        // loses by the larger one's LDS, Conv2d 4 x 62x62x64 -> 384 3x3 132.6 us apart, 142.7 in one launch, and 128 x 64 tiles by
        // an uneven end, 6 x 67x67x64 -> 64 50.9 and 54.0.  Smaller tiles of x's product beside small areas: any number,
        // 64 x 14x14x32 -> 64 5x5 48.0 and 37.1)
        if (tx == TILE_128x32) mx = ceil_div(gx.M, 128), nx = ceil_div(gx.N, 32);
        else grid_of(tx, gx, mx, nx);
        auto long_m = [](TileId t) { return t == TILE_128x128 || t == TILE_128x64 || t == TILE_128x32; };
        auto long_n = [](TileId t) { return t == TILE_128x128 || t == TILE_64x128; };
        const bool rows = long_m(tx) || long_m(ty), cols = long_n(tx) || long_n(ty);
        if ((rows && cols) || (tx != TILE_64x64 && tx != TILE_128x32)) return (long)mx * nx * gx.splits + (long)my * ny * gy.splits <= 2L * cu_count();
    }
    return (long)ceil_div(gx.M, 64) * ceil_div(gx.N, 32) * (gx.virt == VIRT_A_CLASSES ? gx.ncls : gx.splits) + (long)my * ny * gy.splits < 0x7fffffffL;
}

template <typename E, typename X, int EDGE>
static int kept_launch_y(TileId ty, const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    switch (ty) {
        case TILE_128x128: return launch_pair_tiles<X, typename TileOf<E, 128, 128, false, false, VIRT_B_KROWS>::type, EDGE>(gx, gy, stream);
        case TILE_64x128: return launch_pair_tiles<X, typename TileOf<E, 64, 128, false, false, VIRT_B_KROWS>::type, EDGE>(gx, gy, stream);
        default: return launch_pair_tiles<X, typename TileOf<E, 64, 64, false, false, VIRT_B_KROWS>::type, EDGE>(gx, gy, stream);
    }
}

// (a last K step that K cuts short asks nothing of the filter gradient, whose rows end with their buffer)
template <typename E, int VIRT, int EDGE>
static int kept_launch_x(TileId tx, TileId ty, const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    switch (tx) {
        case TILE_64x64:
            if constexpr (VIRT == VIRT_A_ROWS) return kept_launch_y<E, typename TileOf<E, 64, 64, true, false, VIRT>::type, EDGE>(ty, gx, gy, stream);
            break;
        case TILE_64x128:
            if constexpr (VIRT == VIRT_A_ROWS) return kept_launch_y<E, typename TileOf<E, 64, 128, true, false, VIRT>::type, EDGE>(ty, gx, gy, stream);
            break;
        case TILE_128x32:
            if constexpr (sizeof(E) == 4) return kept_launch_y<E, typename TileOf<E, 128, 32, true, false, VIRT>::type, EDGE>(ty, gx, gy, stream);
            break;
        case TILE_128x64: return kept_launch_y<E, typename TileOf<E, 128, 64, true, false, VIRT>::type, EDGE>(ty, gx, gy, stream);
        default: break;
    }
    return kept_launch_y<E, typename TileOf<E, 128, 128, true, false, VIRT>::type, EDGE>(ty, gx, gy, stream);
}

template <typename E, int VIRT>
static int kept_launch(const GemmArgs &gx, const GemmArgs &gy, hipStream_t stream) {
    TileId tx, ty;
    if (!kept_tiles<E>(gx, gy, tx, ty)) return fail(D8_ERR_ARGUMENT, "gemm_tiled_kept_pair_launch: no kernel for this pair of tiles");
    return gx.K % (128 / (int)sizeof(E)) ? kept_launch_x<E, VIRT, EDGE_PIECES>(tx, ty, gx, gy, stream) : kept_launch_x<E, VIRT, EDGE_NONE>(tx, ty, gx, gy, stream);
}

}  // namespace d8

#endif
