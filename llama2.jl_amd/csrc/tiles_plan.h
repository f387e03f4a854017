// How k_tiles.hip deals out the tiles of a product: which workgroup takes what.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

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

// The grouped products' blocks of positions (k_group makes the lists, one for each of the two products of an expert).  A block has `units` of 64 positions, up
// to five; an expert's units go in equal shares to as few blocks as a bound b on them allows, and the bound is the one whose blocks are likely through first.
//
// A tile of 256 rows takes about as long as 18 of its steps of 64 inputs with one unit would on the matrix cores alone (launch, first loads, epilogue), and in
// each step 0.45 us a unit, but no less than its loads do (0.93 and 1.12 us for one and two units where every compute unit has one).  Blocks fall to the compute units in
// rounds.  us, at most 64 / 128 / 192 / 256 / 320 positions a block, and before in blocks of 256 and remainders: 32 experts of 232 to 280, 1024 rows x 2048 inputs 74 / 74 /
// 57 / 70 / 79 (72), 2048 x 1024 72 / 62 / 52 / 66 / 47 (67); gated 4096 x 4096 590 / 436 / 344 / 385 / 299 (400), 4096 x 2048 340 / 237 / 209 / 205 / 177 (210); 16 of
// 69 to 97, 2048 x 4096 54 / 66 / 66 / 66 / 66 (67), 4096 x 2048 56 / 47 / 47 / 47 / 47 (48); 16 of 440 to 560, 2048 x 2048 gated 117 / 107 / 101 / 126 / 85 (130); 8 of 1 to
// 900, 1344 x 1344 23 / 30 / 40 / 51 / 60 (51).
#define TILES_UNIT 64
#define TILES_MAX_UNITS 5
// a / b for a < 2^21 (a + 1/2 is at least 1/2 from a multiple of b, and the product's error less than that: no division where a single workgroup waits for it)
__host__ __device__ inline unsigned tiles_quot(unsigned a, unsigned b) {
#ifdef __HIP_DEVICE_COMPILE__
    return (unsigned)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)b));
#else
    return a / b;
#endif
}
struct TilesSplit {
    unsigned blocks, weight, largest;  // weight: tenths of a unit's step, over the blocks
};
__host__ __device__ inline unsigned tiles_weight(unsigned units) { return units == 1 ? 21 : units == 2 ? 25 : 10 * units; }
// an expert's units in n blocks: block k begins at unit at(k)
struct TilesShares {
    unsigned q, more;
    __host__ __device__ TilesShares(unsigned units, unsigned n) : q(n ? tiles_quot(units, n) : 0), more(units - n * q) {}
    __host__ __device__ unsigned at(unsigned k) const { return k * q + (k < more ? k : more); }
};
__host__ __device__ inline unsigned tiles_blocks(unsigned units, unsigned b) { return tiles_quot(units + b - 1, b); }
// `units` of an expert in blocks of at most b
__host__ __device__ inline TilesSplit tiles_split(unsigned units, unsigned b) {
    const unsigned n = tiles_blocks(units, b);
    const TilesShares s(units, n);
    return {n, s.more * tiles_weight(s.q + 1) + (n - s.more) * tiles_weight(s.q), s.q + (s.more ? 1u : 0u)};
}
// What blocks of at most b units may take with n_nt row groups of `steps` steps on n_cu compute units: half of the experts have a standard deviation
// more of the rows than the others' share, half as much less.  (By what every expert really has, in the launch that counts it: 22 us of that launch's one
// workgroup instead of 9, its code being fetched for the purpose, and the same choice for the cases above.)
inline float tiles_time(double rows, int experts, unsigned b, unsigned n_nt, unsigned steps, unsigned n_cu) {
    const double share = rows / experts, dev = std::sqrt(share);
    double blocks = 0.0, weight = 0.0;
    unsigned largest = 0;
    for (int more = 0; more < 2; more++) {
        const TilesSplit v = tiles_split((unsigned)std::ceil((more ? share + dev : std::max(1.0, share - dev)) / TILES_UNIT), b);
        blocks += 0.5 * experts * v.blocks;
        weight += 0.5 * experts * v.weight;
        largest = std::max(largest, v.largest);
    }
    const double sum = std::ceil(blocks * n_nt / n_cu) * (180.0 + steps * weight / blocks);
    return (float)std::max(sum, 180.0 + (double)steps * tiles_weight(largest));
}
// the bound for `rows` rows in all
inline unsigned tiles_bound(int64_t rows, int experts, unsigned n_nt, unsigned steps, unsigned n_cu) {
    unsigned best = 1;
    for (unsigned b = 2; b <= TILES_MAX_UNITS; b++)
        if (tiles_time((double)rows, experts, b, n_nt, steps, n_cu) < tiles_time((double)rows, experts, best, n_nt, steps, n_cu)) best = b;
    return best;
}
// The bound is made for experts that have about as many rows each.  Where it is more than one, the launch that counts the rows compares it with blocks of whole tiles,
// by the blocks that there really are: few experts may take most.  us, that bound, with this, and blocks of 256 as they come; 16 experts of which two take every one of
// 500 positions, 3584 x 3584 134, 108, 108; four every one of 2000, 2048 x 2048 73, 62, 65, 3584 x 3584 208, 175, 181, 4096 x 4096 232, 195, 203; one of them, 4096 x
// 4096 325, 292, 303; the counting launch 3.4 and 8.7 to 4.1 and 9.4.  (Over 7 shapes, 130 to 2000 positions and 1 to 4 such experts 2 % above blocks of 256 at most, 0.64 to
// 0.79 of their time in the mean; a bound of one is never the slower of those.)
#define TILES_WHOLE_UNITS 4
struct TilesRule {
    unsigned bound, n_nt, steps, n_cu;  // n_cu 0: the bound, whatever the blocks
};
// rounds of the blocks, each of the time of the mean block
__host__ __device__ inline float tiles_rounds(const TilesRule &r, unsigned blocks, unsigned weight) {
    return (float)tiles_quot(blocks * r.n_nt + r.n_cu - 1, r.n_cu) * (180.0f + (float)(r.steps * weight) / (float)blocks);
}

// and the most blocks that there can be
inline int64_t tiles_most(int64_t rows, int experts, unsigned b) {
    return ((rows + TILES_UNIT - 1) / TILES_UNIT + experts) / b + experts;
}

// of a rule that may come to either
inline int64_t tiles_most(int64_t rows, int experts, const TilesRule &r) { return tiles_most(rows, experts, r.n_cu ? std::min(r.bound, (unsigned)TILES_WHOLE_UNITS) : r.bound); }
inline TilesRule tiles_rule(int64_t rows, int experts, unsigned n_nt, unsigned steps, unsigned n_cu) {
    TilesRule r = {tiles_bound(rows, experts, n_nt, steps, n_cu), n_nt, steps, n_cu};
    const int64_t most = tiles_most(rows, experts, 1);
    if (r.bound == 1 || r.bound == TILES_WHOLE_UNITS || most * n_nt + n_cu >= (1 << 21) || most * 25 * steps >= ((int64_t)1 << 31)) r.n_cu = 0;
    return r;
}

// A single product's positions in the same kind of blocks, every row group's alike: the bound for them and what they may take
inline float tiles_cost(unsigned units, unsigned steps) { return 180.0f + (float)(steps * tiles_weight(units)); }
// (whole tiles of 256 positions, and their rest as halves)
inline float tiles_whole_time(const TilesPlan &p, unsigned steps, unsigned n_cu) {
    return (float)((p.whole + n_cu - 1) / n_cu) * tiles_cost(4, steps) + (p.whole < p.n ? tiles_cost(2, steps) : 0.0f);
}
inline float tiles_dense_time(unsigned units, unsigned b, unsigned n_nt, unsigned steps, unsigned n_cu) {
    const TilesSplit v = tiles_split(units, b);
    const float rounds = (float)((v.blocks * n_nt + n_cu - 1) / n_cu), sum = rounds * (180.0f + (float)steps * (float)v.weight / (float)v.blocks);
    return std::max(sum, tiles_cost(v.largest, steps));
}
inline unsigned tiles_dense_bound(unsigned units, unsigned n_nt, unsigned steps, unsigned n_cu) {
    unsigned best = 1;
    for (unsigned b = 2; b <= TILES_MAX_UNITS; b++)
        if (tiles_dense_time(units, b, n_nt, steps, n_cu) <= tiles_dense_time(units, best, n_nt, steps, n_cu)) best = b;
    return best;
}
// block k of `blocks` of a row group's units, item = row group * blocks + k of a grid of tiles_workgroups(items)
struct TilesBlock {
    bool any;
    unsigned nt, at, units;  // at: in units
};
__host__ __device__ inline TilesBlock tiles_block(unsigned units, unsigned blocks, unsigned items, unsigned workgroup) {
    const unsigned item = tiles_deal(items, workgroup);
    if (item >= items) return {false, 0, 0, 0};
    const unsigned nt = item / blocks, k = item - nt * blocks;
    const TilesShares s(units, blocks);
    return {true, nt, s.at(k), s.at(k + 1) - s.at(k)};
}
