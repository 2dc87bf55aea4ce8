// Which pairs of products run longer in one launch than in two (gemm_tiled_pair_plain.h, gemm_tiled_pair_kept.h).
#ifndef DEEP8_AMD_GEMM_TILED_PAIR_TAIL_H
#define DEEP8_AMD_GEMM_TILED_PAIR_TAIL_H

#include "gemm_tiled_kernel.h"

namespace d8 {

static inline int tile_rows(TileId t) { return t == TILE_64x64 || t == TILE_64x128 ? 64 : 128; }
static inline int tile_cols(TileId t) { return t == TILE_128x32 ? 32 : t == TILE_64x64 || t == TILE_128x64 ? 64 : 128; }

// A few workgroups more than the chip holds at once, of products that fill their own rounds: those few start when the long ones before them
// end, and run one to a compute unit.  wg0 and wg1 workgroups; how many a compute unit holds is what the larger sides of the two tiles
// leave of its LDS.  588 drawn pairs of more workgroups than two to a compute unit, 89 of which run more than 3 % longer in one launch: of the
// 55 that the line for two to a compute unit takes out 26 do (2.1 % at the mean, 2 x 97x97x384 -> 192 1x1 74.9 us apart, 80.2 in one launch, Conv2d 1 x
// 88x88x496 -> 64 3x3 88.7 and 96.5), of the 33 that the one for more takes out 12 (1.4 %; 4352 x 448 x 832 60.5 and 68.1).  The others' losses lie
// among gains of the same shapes: on the whole one launch saves 7 %.
static inline bool leaves_a_tail(const GemmArgs &g0, TileId t0, long wg0, const GemmArgs &g1, TileId t1, long wg1) {
    const long cus = cu_count();
    const int rows = tile_rows(t0) > tile_rows(t1) ? tile_rows(t0) : tile_rows(t1), cols = tile_cols(t0) > tile_cols(t1) ? tile_cols(t0) : tile_cols(t1);
    const bool two = rows + cols == 256;
    const double waves = (double)(wg0 + wg1) / ((two ? 2 : rows + cols > 128 ? 3 : 4) * cus);
    auto fill = [&](long wgs) { return (double)wgs / (cus * ((wgs + cus - 1) / cus)); };  // of its own rounds
    auto work = [](const GemmArgs &g, TileId t) {  // of a workgroup, in steps of a 128 x 128 tile
        return (double)(g.splits > 1 ? g.tiles_per_split : g.red * ceil_div(g.K, 32)) * tile_rows(t) * tile_cols(t) / (128 * 128);
    };
    const double least = two ? 0.75 : 0.85, longer = work(g0, t0) > work(g1, t1) ? work(g0, t0) : work(g1, t1);
    return waves > 1.05 && waves <= (two ? 1.5 : 1.25) && fill(wg0) >= least && fill(wg1) >= least && longer >= (two ? 14.0 : 6.0);
}

// The same in half, on tiles of which a compute unit holds two: one product's workgroups are a round by themselves, the other's a few more
// than that.  Of 1170 drawn pairs the line takes out 21, 5 % faster apart at the mean and none more than 1.6 % slower (12 x 192 x 1984 x 2048
// 55.1 us apart, 59.7 in one launch, 7 x 1344 x 400 x 2368 70.1 and 75.5, 2048 x 1856 x 2688 60.1 and 63.2); 3 of the others lose more than 3 %.  Shorter
// workgroups, more pieces (whose passes share a launch too) and fuller second rounds gain.
static inline bool leaves_a_half_tail(const GemmArgs &g0, TileId t0, long wg0, const GemmArgs &g1, TileId t1, long wg1) {
    const int rows = tile_rows(t0) > tile_rows(t1) ? tile_rows(t0) : tile_rows(t1), cols = tile_cols(t0) > tile_cols(t1) ? tile_cols(t0) : tile_cols(t1);
    if (rows + cols != 256 || g0.splits > 3 || g1.splits > 3) return false;
    const double cus = cu_count(), rounds = (wg0 + wg1) / (2.0 * cus), fewer = wg0 < wg1 ? wg0 : wg1;
    auto work = [](const GemmArgs &g, TileId t) {  // of a workgroup, in steps of a 128 x 128 tile (half waits for its loads)
        return (double)(g.splits > 1 ? g.tiles_per_split : (long)g.red * ceil_div(g.K, 64)) * (tile_rows(t) + tile_cols(t)) / 256;
    };
    return rounds > 1.0 && rounds <= 1.14 && fewer >= 0.87 * cus && fewer <= cus && work(g0, t0) >= 16.0 && work(g1, t1) >= 16.0;
}

}  // namespace d8

#endif
