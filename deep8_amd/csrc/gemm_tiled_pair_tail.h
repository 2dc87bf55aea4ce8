// Which pairs of products run longer in one launch than in two (gemm_tiled_pair_plain.h, gemm_tiled_pair_kept.h).
#ifndef DEEP8_AMD_GEMM_TILED_PAIR_TAIL_H
#define DEEP8_AMD_GEMM_TILED_PAIR_TAIL_H

#include "gemm_tiled_kernel.h"

namespace d8 {

static inline int tile_rows(TileId t) { return t == TILE_64x64 || t == TILE_64x128 ? 64 : 128; }
static inline int tile_cols(TileId t) { return t == TILE_128x32 ? 32 : t == TILE_64x64 || t == TILE_128x64 ? 64 : 128; }

// A few workgroups more than the chip holds at once, of products that fill their own rounds: those few start when the shorter ones before them
// end, beside long ones that have not, and end behind them.  wg0 and wg1 workgroups; how many a compute unit holds is what the larger sides of the
// two tiles leave of its LDS.  1560 drawn pairs of more workgroups than two to a compute unit, 79 of which run more than 3 % longer in one launch: of
// the 53 that the line takes out 44 do (6.5 % at the mean: 4352 x 448 x 832 60.5 us apart, 68.1 in one launch, Conv2d 2 x 97x97x384 -> 192 1x1 74.9 and
// 80.2) and two are more than 3 % faster together.  The others' losses lie among gains of the same shapes: on the whole one launch saves 9 %.  What it
// leaves out gains: lengths that are nearly the same or three times each other's, exact rounds, long workgroups of 64 x 64 tiles (which wait
// less for each other) that are many steps or leave compute units free, short others where three or four fit.
static inline bool leaves_a_tail(const GemmArgs &g0, TileId t0, long wg0, const GemmArgs &g1, TileId t1, long wg1) {
    const long cus = cu_count();
    const int rows = tile_rows(t0) > tile_rows(t1) ? tile_rows(t0) : tile_rows(t1), cols = tile_cols(t0) > tile_cols(t1) ? tile_cols(t0) : tile_cols(t1);
    const bool two = rows + cols == 256;
    const double waves = (double)(wg0 + wg1) / ((two ? 2 : rows + cols > 128 ? 3 : 4) * cus);
    auto fill = [&](long wgs) { return (double)wgs / (cus * ((wgs + cus - 1) / cus)); };  // of its own rounds
    auto work = [](const GemmArgs &g, TileId t) {  // of a workgroup, in steps of a 128 x 128 tile
        return (double)(g.splits > 1 ? g.tiles_per_split : g.red * ceil_div(g.K, 32)) * tile_rows(t) * tile_cols(t) / (128 * 128);
    };
    const bool first = work(g0, t0) > work(g1, t1);  // whose workgroups are the longer ones
    const double longer = first ? work(g0, t0) : work(g1, t1), shorter = first ? work(g1, t1) : work(g0, t0), least = two ? 0.75 : 0.83;
    if (waves <= 1.05 || waves > (two ? 1.49 : 1.25) || fill(wg0) < least || fill(wg1) < least || longer < 1.25 * shorter || longer >= 3.0 * shorter) return false;
    if (!two) return longer >= 6.0 && shorter >= 3.5;
    const long wgs = first ? wg0 : wg1;
    const bool small = (first ? t0 : t1) == TILE_64x64, many = small && ((first ? g0 : g1).splits > 4 || longer > 25.0 || fill(wgs) < 0.89);
    return longer >= 14.0 && wgs % cus != 0 && !many && t0 != TILE_128x32 && t1 != TILE_128x32;
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
