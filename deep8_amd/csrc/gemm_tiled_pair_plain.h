// Two real products as one launch of the tiled kernel (gemm_tiled_pair_kernel, gemm_tiled_kernel.h): the two gradients of a
// mid-size MatrixMultiply.  Included by the translation units that instantiate it.
#ifndef DEEP8_AMD_GEMM_TILED_PAIR_PLAIN_H
#define DEEP8_AMD_GEMM_TILED_PAIR_PLAIN_H

#include "gemm_tiled_pair_tail.h"

namespace d8 {

// g0 is NT (a MatrixMultiply's gradient of its first input),
// g1 is TN (the gradient of its second); either may be batched or split along its reduction (the caller reduces).
template <typename E>
static bool plain_pair_tiles(const GemmArgs &g0, const GemmArgs &g1, TileId &t0, TileId &t1) {
    t0 = choose_tile<E, true, true>(g0), t1 = choose_tile<E, false, false>(g1);
    auto ok = [](TileId t) { return t == TILE_64x128 || t == TILE_128x128 || t == TILE_128x64 || t == TILE_64x64; };
    return ok(t0) && ok(t1) && g0.packed == g1.packed;
}

template <typename E, int EDGE>
static int launch_plain_pair(const GemmArgs &g0, const GemmArgs &g1, hipStream_t stream) {
    TileId t0, t1;
    if (!plain_pair_tiles<E>(g0, g1, t0, t1)) return fail(D8_ERR_ARGUMENT, "gemm_tiled_plain_pair_launch: no kernel for this pair of tiles");
#define D8_PAIR_1(T0T)                                                                                              \
    switch (t1) {                                                                                                   \
        case TILE_128x128: return launch_pair_tiles<T0T, typename TileOf<E, 128, 128, false, false>::type, EDGE>(g0, g1, stream);    \
        case TILE_64x128: return launch_pair_tiles<T0T, typename TileOf<E, 64, 128, false, false>::type, EDGE>(g0, g1, stream);      \
        case TILE_64x64: return launch_pair_tiles<T0T, typename TileOf<E, 64, 64, false, false>::type, EDGE>(g0, g1, stream);        \
        default: return launch_pair_tiles<T0T, typename TileOf<E, 128, 64, false, false>::type, EDGE>(g0, g1, stream);               \
    }
    typedef typename TileOf<E, 64, 128, true, true>::type A0;
    typedef typename TileOf<E, 128, 128, true, true>::type A1;
    typedef typename TileOf<E, 128, 64, true, true>::type A2;
    typedef typename TileOf<E, 64, 64, true, true>::type A3;
    if (t0 == TILE_64x64) { D8_PAIR_1(A3) }
    if (t0 == TILE_64x128) { D8_PAIR_1(A0) }
    if (t0 == TILE_128x128) { D8_PAIR_1(A1) }
    D8_PAIR_1(A2)
#undef D8_PAIR_1
}

}  // namespace d8

#endif
