// The band bookkeeping of the ScanND forward's host side over long and short
// 3D grids, in the order in which a launch runs it: the tile rule, then the
// tiles of every band. Built with the address sanitizer; the tables have
// exactly the entries of the library's.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "scannd_tiles.hpp"

int main() {
    const int lead_axis[] = {1, 2, 7, 60, 400, 1500, 1535, 1536, 1540, 3072, 3080, 8000, 8190, 8192, 8200, 12000, 16380};
    const int rows[] = {1, 3, 4, 7, 8, 13, 16}, cols[] = {1, 8, 17, 64};
    int checked = 0, took_small = 0;
    for (int order = 0; order < 3; ++order)
        for (int n : lead_axis)
            for (int r : rows)
                for (int c : cols) {
                    int dims[3] = {n, r, c};
                    std::swap(dims[0], dims[order]);
                    int tile[3], ntile[3];
                    if (km::nd_tiles(3, dims, 8, 4, tile, ntile) > km::kMaxBands) continue;
                    const bool small = km::nd_small_tiles(dims, 8, 1, SIZE_MAX, tile, ntile);
                    if (!small) km::nd_tiles(3, dims, 8, 4, tile, ntile);
                    long nbands = 1, want = 1;
                    for (int ax = 0; ax < 3; ++ax) {
                        nbands += ntile[ax] - 1;
                        want *= ntile[ax];
                    }
                    std::vector<long> cnt(km::kMaxBands), nxt(km::kMaxBands);
                    const long n_tiles = km::nd_band_counts(3, ntile, cnt.data(), nxt.data());
                    long sum = 0;
                    for (long b = 0; b < nbands; ++b) sum += cnt.at(b);
                    if (n_tiles != want || sum != want) {
                        std::printf("%dx%dx%d: %ld tiles counted, %ld in bands, %ld exist\n", dims[0], dims[1], dims[2],
                                    n_tiles, sum, want);
                        return 1;
                    }
                    // Without a band table a launch per band would follow.
                    if (small && nbands > km::kMaxFlowBands) {
                        std::printf("%dx%dx%d: small tiles in %ld bands\n", dims[0], dims[1], dims[2], nbands);
                        return 1;
                    }
                    ++checked;
                    took_small += small;
                }
    // Both sides of the rule, as they measured.
    const int faster[][3] = {{700, 8, 8}, {8, 8, 600}, {7, 7, 60}, {100, 9, 8}, {32, 32, 32}, {20, 19, 23}};
    const int slower[][3] = {{400, 7, 8}, {60, 7, 7}, {100, 7, 16}, {3, 4, 5}, {100, 3, 3}, {2000, 8, 8}, {9, 3, 4}, {6, 2, 2}, {30, 3, 16}};
    int tile[3], ntile[3];
    for (const auto &d : faster)
        if (!km::nd_small_tiles(d, 8, 16, SIZE_MAX, tile, ntile)) return std::printf("%dx%dx%d\n", d[0], d[1], d[2]);
    for (const auto &d : slower)
        if (km::nd_small_tiles(d, 8, 16, SIZE_MAX, tile, ntile)) return std::printf("%dx%dx%d\n", d[0], d[1], d[2]);
    // More bands than entries are refused, not written.
    const int many[3] = {3000, 1500, 1};
    std::vector<long> cnt(km::kMaxBands), nxt(km::kMaxBands);
    if (km::nd_band_counts(3, many, cnt.data(), nxt.data()) != 0) return 1;
    std::printf("%d grids, %d on small tiles\n", checked, took_small);
    return checked > 500 && took_small > 100 ? 0 : 1;
}
