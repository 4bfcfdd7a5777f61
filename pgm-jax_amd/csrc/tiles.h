// tiles.h -- the tiles of the PME grid and the offsets of their blocks (host code, plain C++).
#pragma once

#include <algorithm>
#include <vector>

namespace pgm {

struct PMETiles {
    int T[3];    // tile width per axis (the last tile may be narrower, >= P-1)
    int nt[3];   // tiles per axis
    int nc[3];   // cubes of 2 x 2 x 2 tiles per axis: (nt + 1) / 2
    int ncubes;  // nc0 nc1 nc2
    int ntiles;  // 8 ncubes: tiles by fine key (octants past the grid stay empty)
    int B[3];    // extent of a tile's block per axis: T + P - 1
    int bsize;   // values stored per block: B0 B1 PME_ZROW
};

// z rows of the stored spread blocks: padded to 16 values, so that a row is one aligned segment and one
// column block of the matrix instructions.
constexpr int PME_ZROW = 16;

constexpr unsigned PME_NO_BLOCK = ~0u;  // merge table: no second block covers the point
constexpr int PME_MAX_CUBES = 1023;     // per axis: ten bits of a packed cube coordinate

// Tiles of a grid of K points per axis at order P: per axis the largest T in cap..P-1 with at least three
// tiles and a last tile at least P-1 wide, numbered in cubes of 2 x 2 x 2 tiles.  False where there is no such
// T or where the blocks hold more values than the merge table's 32-bit offsets reach (768^3 points at order
// 6 hold 2.4e9, 928^3 4.2e9).
inline bool pme_tiles(const int *K, int P, int cap, PMETiles &t) {
    long long cubes = 1;
    for (int a = 0; a < 3; ++a) {
        int best = 0;
        for (int T = cap; T >= P - 1 && !best; --T) {
            const int nt = (K[a] + T - 1) / T;
            const int last = K[a] - (nt - 1) * T;
            if (nt >= 3 && last >= P - 1) best = T;
        }
        if (!best) return false;
        t.T[a] = best;
        t.nt[a] = (K[a] + best - 1) / best;
        t.nc[a] = (t.nt[a] + 1) / 2;
        t.B[a] = best + P - 1;
        if (t.nc[a] > PME_MAX_CUBES) return false;
        cubes *= t.nc[a];
    }
    t.bsize = t.B[0] * t.B[1] * PME_ZROW;
    if (8 * cubes * t.bsize >= (long long)PME_NO_BLOCK) return false;
    t.ncubes = (int)cubes;
    t.ntiles = 8 * t.ncubes;
    return true;
}

// The merge table of the tiles (k_merge_table): per axis and grid coordinate g the offset of the point in its own
// tile's block and in the previous tile's, PME_NO_BLOCK where that does not reach it.
inline std::vector<unsigned> pme_merge_table(const int *K, int P, const PMETiles &t) {
    std::vector<unsigned> tab;
    for (int a = 0; a < 3; ++a) {
        const int T = t.T[a], nt = t.nt[a];
        const int stride = a == 0 ? t.B[1] * PME_ZROW : (a == 1 ? PME_ZROW : 1);
        const unsigned cube = 8 * (a == 0 ? t.nc[1] * t.nc[2] : (a == 1 ? t.nc[2] : 1)), oct = 4 >> a;
        const auto A = [&](int u) { return ((u >> 1) * cube + (u & 1) * oct) * (unsigned)t.bsize; };
        for (int g = 0; g < K[a]; ++g) {
            const int u = std::min(g / T, nt - 1), l = g - u * T;
            tab.push_back(A(u) + l * stride);
            if (l <= P - 2) {
                const int up = u > 0 ? u - 1 : nt - 1;
                const int width = up < nt - 1 ? T : K[a] - (nt - 1) * T;
                tab.push_back(A(up) + (l + width) * stride);
            } else {
                tab.push_back(PME_NO_BLOCK);
            }
        }
    }
    return tab;
}

}  // namespace pgm
