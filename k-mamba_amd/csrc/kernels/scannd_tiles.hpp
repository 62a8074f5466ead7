// scannd_tiles.hpp - the tilings of the ScanND forward's grids: tiles per
// axis, tiles per band, and the rule for small 3D grids. Host code without
// HIP, so that a CPU program can check it.
#pragma once

#include <algorithm>
#include <cstddef>

namespace km {

// Bands a launch per band may have, and the dataflow schedule's band table
// (a kernel argument) holds.
constexpr long kMaxBands = 4096;
constexpr int kMaxFlowBands = 768;

// Tiles of `row` points along the last axis and `lead` along each leading
// axis; returns the bands (sums of tile indices). The kernels prefetch rows one
// ahead, so every tile needs at least two rows per plane below an in-tile
// leading axis: the row-axis tile grows while its last tile would hold one row,
// and tiles are 1 along the leading axes when the row axis has length 1.
inline long nd_tiles(int nd, const int *dims, int row, int lead, int *tile, int *ntile) {
    const int rax = nd - 2;
    int trow = std::min(dims[rax], lead);
    while (trow < dims[rax] && dims[rax] % trow == 1) ++trow;
    long nbands = 1;
    for (int ax = 0; ax < nd; ++ax) {
        int t = ax == nd - 1 ? row : ax == rax ? trow : lead;
        if (ax < rax && dims[rax] == 1) t = 1;
        tile[ax] = std::min(dims[ax], t);
        ntile[ax] = (dims[ax] + tile[ax] - 1) / tile[ax];
        nbands += ntile[ax] - 1;
    }
    return nbands;
}

// Tiles per band, the distribution of tile-index sums, into cnt (nxt is
// scratch; both of kMaxBands entries). Returns the tiles, or 0 when there are
// more bands than entries.
inline long nd_band_counts(int nd, const int *ntile, long *cnt, long *nxt) {
    long nbands = 1, n = 1;
    for (int ax = 0; ax < nd; ++ax) {
        nbands += ntile[ax] - 1;
        n *= ntile[ax];
    }
    if (nbands > kMaxBands) return 0;
    cnt[0] = 1;
    long reach = 0;
    for (int ax = 0; ax < nd; ++ax) {
        for (long i = 0; i <= reach + ntile[ax] - 1; ++i) nxt[i] = 0;
        for (long i = 0; i <= reach; ++i)
            for (int v = 0; v < ntile[ax]; ++v) nxt[i + v] += cnt[i];
        reach += ntile[ax] - 1;
        for (long i = 0; i <= reach; ++i) cnt[i] = nxt[i];
    }
    return n;
}

// 3D under the dataflow schedule: a small grid leaves the chip idle while 4 x
// 4 x 8 sub-tiles hand over from one to the next, so it takes tiles of 2 x 2 x
// 8 while their average front (tiles / bands, a wave per channel group each) is
// below three quarters of a wave per SIMD; above, the pencils' ring, which
// reads less back, wins. M = 16, pencils / small tiles (us), by that front:
// 20x17x23 D64 (216) 218 / 155, 32x32x32 D64 (482) 378 / 293, 48x20x40 D64
// (519) 420 / 318, 6x60x60 D128 (591) 530 / 327, 32x32x32 D96 (723) 405 / 371,
// 40x40x40 D64 (744) 525 / 476, 40x30x36 D112 (1105) 541 / 614, 50x50x50 D64
// (1272) 779 / 932. Both are 8 points wide, so y's sums keep their order.
// (Width 4 was faster still, 133 and 441, 984 on the first, second and last but
// one, but changes it.)
constexpr long kSmallFront = 768;
// The critical path of a tiling (us): its fronts, each a hand-over and the
// tile's rows of 8 points one after the other. Smaller tiles shorten it where
// they split a plane, not where they only split axis 0 (an axis of 3 or 7 rows
// is one tile, or two of 4, either way), and not on a grid of one column of
// tiles, whose pencil hands nothing over. M = 16, D64, pencils / small tiles:
// 700x8x8 3270 / 2035, 8x8x600 1490 / 520, but 400x7x8 1850 / 2005, 100x3x3 320
// / 357, 60x7x7 296 / 312; 9x3x4 D320 M = 1 36.5 / 39.2. (By 5 %: the model's
// error; 30x3x16 D64, 2 % shorter by it, 119 / 129.)
inline double nd_path_us(long nbands, const int *tile) { return nbands * (1.6 + 1.05 * tile[0] * tile[1]); }
// Sets tile and ntile to the 2 x 2 x `row` tiles (axis 1 may have more rows,
// see nd_tiles) and returns true where they are the faster ones for ncg channel
// groups, their flags fit max_flags and their bands, about twice those of the
// larger tiles (whose pencils leave axis 0 out), fit the dataflow schedule's
// table: without it they would run a launch per band (1600x16x16 D128, M = 16:
// 16940 us, on pencils 9220; 2000x8x8 D64: 23490 and 9210).
inline bool nd_small_tiles(const int *dims, int row, long ncg, size_t max_flags, int *tile, int *ntile) {
    int tile4[3], ntile4[3];
    const double path4 = nd_path_us(nd_tiles(3, dims, row, 4, tile4, ntile4), tile4);
    const long nbands = nd_tiles(3, dims, row, 2, tile, ntile);
    const long n = static_cast<long>(ntile[0]) * ntile[1] * ntile[2] * ncg;
    return nbands <= kMaxFlowBands && n <= kSmallFront * nbands && nd_path_us(nbands, tile) < 0.95 * path4 &&
           ntile[1] * ntile[2] > 1 && static_cast<size_t>(n) <= max_flags;
}

}  // namespace km
