// The launch of one product on the tile its shape asks for.  Included by the translation units that instantiate the tiled
// kernels: one per element type and kind of operands, so that they compile side by side.
#ifndef DEEP8_AMD_GEMM_TILED_LAUNCH_H
#define DEEP8_AMD_GEMM_TILED_LAUNCH_H

#include "gemm_tiled_kernel.h"

namespace d8 {

template <typename T>
static constexpr long lds_bytes() {
    if constexpr (T::DMA) return T::LDS_BYTES;
    else return 2L * (T::A_SZ + T::B_SZ) * T::ES;
}

template <typename T, int EDGE>
static int launch_edge(const GemmArgs &g0, hipStream_t stream) {
    GemmArgs g = g0;
    constexpr int BM = T::BM, BN = T::BN, VIRT = T::VIRT;
    const bool tail = g.tail_splits > 0;  // (gemm_tiled_run sets it only for 128-row tiles and a tail_m0 that is a multiple of them)
    const int tilesM = ceil_div(tail ? g.tail_m0 : g.M, BM), tilesN = ceil_div(g.N, BN);
    const int extra = tail ? ceil_div(g.M - g.tail_m0, BM) * tilesN * g.tail_splits : 0;
    // A launch of at most two workgroups per CU is spread evenly only if a CU cannot take a third:
    // where the tile's own LDS would let three in, unused dynamic LDS is requested on top.
    constexpr long lds = lds_bytes<T>(), third = 160 * 1024 / 3;
    const int layers = VIRT == VIRT_A_CLASSES ? g.ncls : g.batch * g.splits;  // for classes g.M is the largest one's
    const long wgs = (long)tilesM * tilesN * layers, cus = cu_count();
    const unsigned pad = (lds <= third && wgs > cus && wgs <= 2 * cus) ? (unsigned)(third + 512 - lds) : 0u;
    // a launch whose records would not fit the caller's buffer writes none
    g.phase_rec = (size_t)(tilesM * tilesN + extra) * layers * 64 <= phase_rec_bytes ? phase_rec_buf : nullptr;
    set_reciprocals(g, tilesM, tilesN, BM, T::BK, tilesM * tilesN + extra);
    const dim3 grid(tilesM * tilesN + extra, 1, layers);
    hipLaunchKernelGGL((gemm_tiled_kernel<T, EDGE>), grid, dim3(T::NT), pad, stream, g, tilesM, tilesN);
    D8_LAUNCH_CHECK();
    return 0;
}

template <typename T>
static int launch_whole(const GemmArgs &g, hipStream_t stream) {
    if constexpr (T::DMA && T::VIRT == VIRT_NONE)
        if (g.packed) return launch_edge<T, EDGE_ANY>(g, stream);
    if constexpr (T::VIRT != VIRT_B_KROWS)
        if (g.K % T::BK) return launch_edge<T, EDGE_PIECES>(g, stream);
    return launch_edge<T, EDGE_NONE>(g, stream);
}

template <typename E, int BM, int BN, bool A_KC, bool B_KC, int VIRT>
static int launch_tiled(const GemmArgs &g, hipStream_t stream, bool any = false) {
    if constexpr (VIRT == VIRT_NONE && BM <= 128)  // rows that start anywhere: shifted into place between memory and LDS
        if (any) return launch_edge<Tile<E, BM, BN, BN == 32 ? 4 : 2, BN == 32 ? 1 : 2, A_KC, B_KC, VIRT>, EDGE_ANY>(g, stream);
    if constexpr (sizeof(E) == 2 && BM <= 128) {
        const long wgs = (long)ceil_div(g.M, BM) * ceil_div(g.N, BN) * (VIRT == VIRT_A_CLASSES ? g.ncls : g.batch * g.splits);
        if constexpr (BM == 128 && BN == 128) {
            if (wgs <= cu_count()) return launch_whole<typename TileOf<E, BM, BN, A_KC, B_KC, VIRT, 1>::type>(g, stream);
        } else if constexpr (A_KC) {  // (other reductions run over rows or pixels: seldom of few steps, and cut into pieces for the chip)
            typedef typename TileOf<E, BM, BN, A_KC, B_KC, VIRT, 3>::type T;
            if (wgs > 2L * cu_count() && !g.packed) return g.K % T::BK ? launch_edge<T, EDGE_PIECES>(g, stream) : launch_edge<T, EDGE_NONE>(g, stream);
        }
    }
    return launch_whole<typename TileOf<E, BM, BN, A_KC, B_KC, VIRT>::type>(g, stream);
}

template <typename E, bool A_KC, bool B_KC, int VIRT = VIRT_NONE>
static int pick_tile(const GemmArgs &g, hipStream_t stream) {
    const bool any = VIRT == VIRT_NONE && !in_pieces<E>(g, A_KC, B_KC);
    switch (choose_tile<E, A_KC, B_KC, VIRT>(g, any)) {
        case TILE_WIDE: return gemm_wide_launch(g, !A_KC, B_KC, stream);
        case TILE_256:
            if constexpr (sizeof(E) == 2) return launch_tiled<E, 256, 256, A_KC, B_KC, VIRT>(g, stream);
            break;
        case TILE_128x64: return launch_tiled<E, 128, 64, A_KC, B_KC, VIRT>(g, stream, any);
        case TILE_64x64: return launch_tiled<E, 64, 64, A_KC, B_KC, VIRT>(g, stream, any);
        case TILE_128x32:
            if constexpr (VIRT != VIRT_B_KROWS && sizeof(E) == 4) return launch_tiled<E, 128, 32, A_KC, B_KC, VIRT>(g, stream, any);
            break;
        case TILE_64x128: return launch_tiled<E, 64, 128, A_KC, B_KC, VIRT>(g, stream, any);
        default: break;
    }
    return launch_tiled<E, 128, 128, A_KC, B_KC, VIRT>(g, stream, any);
}

// Real matrices as both operands.
template <typename E>
static int launch_plain(const GemmArgs &g, int transA, int transB, hipStream_t stream) {
    if (!transA && !transB) return pick_tile<E, true, false>(g, stream);
    if (!transA && transB) return pick_tile<E, true, true>(g, stream);
    return pick_tile<E, false, false>(g, stream);
}

// A patch matrix as one of them.
template <typename E>
static int launch_patch(const GemmArgs &g, int transB, hipStream_t stream) {
    if (g.virt == VIRT_A_CLASSES) {  // (the last tile of a class, or its only one, may reach past it)
        if constexpr (sizeof(E) == 4)
            if (g.N <= 32)  // (see narrow_output in gemm.hip)
                return transB ? launch_tiled<E, 128, 32, true, true, VIRT_A_CLASSES>(g, stream)
                              : launch_tiled<E, 128, 32, true, false, VIRT_A_CLASSES>(g, stream);
        if (transB) {
            if (g.N < 128) return launch_tiled<E, 128, 64, true, true, VIRT_A_CLASSES>(g, stream);
            return launch_tiled<E, 128, 128, true, true, VIRT_A_CLASSES>(g, stream);
        }
        if (g.N < 128) return launch_tiled<E, 128, 64, true, false, VIRT_A_CLASSES>(g, stream);
        return launch_tiled<E, 128, 128, true, false, VIRT_A_CLASSES>(g, stream);
    }
    if (g.virt == VIRT_A_ROWS) return transB ? pick_tile<E, true, true, VIRT_A_ROWS>(g, stream) : pick_tile<E, true, false, VIRT_A_ROWS>(g, stream);
    return pick_tile<E, false, false, VIRT_B_KROWS>(g, stream);
}

}  // namespace d8

#endif
