// How k_tiles.hip deals out the tiles of a product: which workgroup takes what.
#pragma once

#include <hip/hip_runtime.h>

// n items go to 8 ceil(n / 8) workgroups, contiguous runs of them to each of the 8 XCDs (to which workgroups go in turn): workgroup b's item, or n and
// beyond where it has none
__host__ __device__ inline unsigned tiles_deal(unsigned n, unsigned b) {
    const unsigned per = (n + 7) / 8;
    return (b >> 3) < per ? (b & 7u) * per + (b >> 3) : n;
}
inline unsigned tiles_workgroups(unsigned n) { return 8 * ((n + 7) / 8); }

// A single product of tiles of 256 positions: the first `whole` of its n tiles as they are, by the workgroups below halves_from; the others as two halves
// of 128 positions each, by those from there on.
struct TilesPlan {
    unsigned n, whole, halves_from;
};
inline unsigned tiles_grid(const TilesPlan &p) { return p.halves_from + tiles_workgroups(2 * (p.n - p.whole)); }
struct TilesWork {
    bool any;
    unsigned item;
    int half;  // 0, 1; -1: the whole tile
};
__host__ __device__ inline TilesWork tiles_work(const TilesPlan &p, unsigned b) {
    if (b < p.halves_from) {
        const unsigned i = tiles_deal(p.whole, b);
        return {i < p.whole, i, -1};
    }
    const unsigned n = 2 * (p.n - p.whole), i = tiles_deal(n, b - p.halves_from);
    return {i < n, p.whole + i / 2, (int)(i & 1u)};
}

// 896 tiles of 28 672 x 4096 over 2048 positions take 465 us in four rounds of 256 compute units, the last half empty, 431 as three rounds and
// 256 halves.  Only where the halves are one round: two rounds of halves take as long as one of whole tiles.
inline TilesPlan tiles_plan(unsigned n, bool halves, int n_cu) {
    const unsigned rest = n % (unsigned)n_cu;
    const unsigned whole = halves && n > rest && rest > 0 && 2 * rest <= (unsigned)n_cu ? n - rest : n;
    return {n, whole, tiles_workgroups(whole)};
}
