// Both gradients of a convolution as one launch (gemm_tiled_pair_kernel, gemm_tiled_kernel.h), each tiled and cut as it would be
// alone: K may cut gx's last step short and either may be split along its reduction (the caller reduces).  gx has patch rows as A
// or runs over the classes of output pixels.  Included by the translation units that instantiate it, one per element type.
#ifndef DEEP8_AMD_GEMM_TILED_PAIR_KEPT_H
#define DEEP8_AMD_GEMM_TILED_PAIR_KEPT_H

#include "gemm_tiled_pair_tail.h"

namespace d8 {

template <typename E>
static SharedLaunch kept_tiles(const GemmArgs &gx, const GemmArgs &gy, TileId &tx, TileId &ty) {
    if (gy.virt != VIRT_B_KROWS || gx.batch != 1 || gy.batch != 1 || gx.tail_splits || gy.tail_splits) return APART;
    if (gx.virt == VIRT_A_CLASSES) {  // (the tiles of gemm_tiled_launch.h)
        if (gx.splits != 1) return APART;
        tx = sizeof(E) == 4 && gx.N <= 32 ? TILE_128x32 : gx.N < 128 ? TILE_128x64 : TILE_128x128;
    } else if (gx.virt == VIRT_A_ROWS) {
        tx = choose_tile<E, true, false, VIRT_A_ROWS>(gx);
    } else {
        return APART;
    }
    ty = choose_tile<E, false, false, VIRT_B_KROWS>(gy);
    const bool x_ok = tx == TILE_64x64 || tx == TILE_64x128 || tx == TILE_128x128 || tx == TILE_128x64 || (sizeof(E) == 4 && tx == TILE_128x32);
    if (!x_ok || (ty != TILE_128x128 && ty != TILE_64x128 && ty != TILE_64x64)) return APART;
    int mx, nx, my, ny;
    grid_of(ty, gy, my, ny);
    if (tx == TILE_128x32) mx = ceil_div(gx.M, 128), nx = ceil_div(gx.N, 32);
    else grid_of(tx, gx, mx, nx);
    const long wx = (long)mx * nx * (gx.virt == VIRT_A_CLASSES ? gx.ncls : gx.splits), wy = (long)my * ny * gy.splits;
    if (wx + wy >= 0x7fffffffL) return APART;
    if (sizeof(E) == 4 && gx.virt == VIRT_A_ROWS) {
        auto long_m = [](TileId t) { return t == TILE_128x128 || t == TILE_128x64 || t == TILE_128x32; };
        auto long_n = [](TileId t) { return t == TILE_128x128 || t == TILE_64x128; };
        const bool rows = long_m(tx) || long_m(ty), cols = long_n(tx) || long_n(ty), both = tx == TILE_128x128 && ty == TILE_128x128;
        // fp32, more workgroups than two to a compute unit, of which smaller tiles would have three, or 128 x 128 tiles in both: as long
        // as no workgroup runs longer than 24 steps of a 128 x 128 tile would (the longer workgroups start first: launch_pair_tiles).
        // 90 drawn layers apart 9351 us, in one launch 9205 without that line; 7 x 35x35x64 -> 64 5x5 50.4 / 40.4, 17 x 17x17x200 -> 148
        // 100 / 85.5, and of longer workgroups DeConv2d 27 x 21x21x320 -> 64 4x4 stride 2 217 / 187, but Conv2d 1 x 93x54x320 -> 64 5x5 107 /
        // 117, 4 x 82x82x64 -> 168 148 / 157.  And none that leaves a tail behind (leaves_a_tail).
        // (Smaller tiles of x's product beside small areas: any number, 64 x 14x14x32 -> 64 5x5 48.0 and 37.1.)
        if (both || (((rows && cols) || (tx != TILE_64x64 && tx != TILE_128x32)) && wx + wy > 2L * cu_count())) {
            auto work = [](const GemmArgs &g, long m, long n) {
                return (g.splits > 1 ? g.tiles_per_split : (long)g.red * ceil_div(g.K, 32)) * m * n;
            };
            const long most = 24 * 128 * 128;
            const bool brief = work(gx, long_m(tx) ? 128 : 64, tx == TILE_128x32 ? 32 : long_n(tx) ? 128 : 64) <= most && work(gy, long_m(ty) ? 128 : 64, long_n(ty) ? 128 : 64) <= most;
            return brief && !leaves_a_tail(gx, tx, wx, gy, ty, wy) ? SHARED_KEPT : APART;
        }
    }
    return SHARED;
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
    if (kept_tiles<E>(gx, gy, tx, ty) == APART) return fail(D8_ERR_ARGUMENT, "gemm_tiled_kept_pair_launch: no kernel for this pair of tiles");
    return gx.K % (128 / (int)sizeof(E)) ? kept_launch_x<E, VIRT, EDGE_PIECES>(tx, ty, gx, gy, stream) : kept_launch_x<E, VIRT, EDGE_NONE>(tx, ty, gx, gy, stream);
}

}  // namespace d8

#endif
