// How k_delta.hip lays out the ring of convolution inputs and takes a prompt's chunks: the record of a chunk, and the chunks whose records lie in memory together.
#pragma once

#include <algorithm>

#include "layered.h"

// The ring of convolution inputs has `taps` slots; a token's step writes slot now = pos % taps while other workgroups read those of the j-th token
// before it (1 <= j; -1: there is none).
__host__ __device__ inline int delta_ring_slot(int taps, int now, int j) { return j >= taps ? -1 : now - j < 0 ? now - j + taps : now - j; }

#define WK_T 32  // tokens of a chunk

// the record of one (chunk, head), NT tiles of 16 key channels (a multiple of 4) and NC of 16 value columns, in words of [64 lanes][4]:
// kt, qt [2 tiles of tokens][NT]; kh [NT][2]; B [3: first, second, second x first tile]; U (before the walk, T V) [NC][2]; S0 [NC][NT]; then
// exp(G_31) [16 NT]
struct DeltaRec {
    int NT, NC;
    __host__ __device__ DeltaRec(int nt, int V) : NT(nt), NC((V + 15) / 16) {}
    __host__ __device__ int kt(int tile, int i) const { return 256 * (tile * NT + i); }
    __host__ __device__ int qt(int tile, int i) const { return 256 * ((2 + tile) * NT + i); }
    __host__ __device__ int kh(int i, int tile) const { return 256 * (4 * NT + 2 * i + tile); }
    __host__ __device__ int b(int i) const { return 256 * (6 * NT + i); }
    __host__ __device__ int u(int c, int tile) const { return 256 * (6 * NT + 3 + 2 * c + tile); }
    __host__ __device__ int s0(int c, int i) const { return 256 * (6 * NT + 3 + 2 * NC + c * NT + i); }
    __host__ __device__ int gc() const { return 256 * (6 * NT + 3 + 2 * NC + NC * NT); }
    __host__ __device__ int floats() const { return gc() + 16 * NT; }
};
inline DeltaRec delta_rec(const DeltaShape &d) { return DeltaRec((d.D + 63) / 64 * 4, d.V); }
inline int64_t delta_chunk_floats(const DeltaShape &d) { return (int64_t)d.H * delta_rec(d).floats(); }  // a chunk's, of all heads

#define DELTA_CHUNK16 16  // tokens of a chunk of the other form, and its record
__host__ __device__ inline int64_t delta_rec16_floats(int NT) { return (int64_t)NT * 784 + 512; }
inline int64_t delta_rec16_floats(const DeltaShape &d, int M) {
    return (int64_t)((M + DELTA_CHUNK16 - 1) / DELTA_CHUNK16) * d.H * delta_rec16_floats(delta_rec(d).NT);
}

// Chunks of 32 or of 16.  The first walk half as many, with less on the chain, but leave the state before every chunk in memory (8 bytes of its element
// written and read, where the other form's outputs are 8 bytes of a row's), and their outputs' workgroups have a head's whole row of values each.  So they pay while
// the walk's latency is what there is to gain: with a state of up to 3 MB in all (2 MB above 128 key channels, whose operands leave a SIMD one wavefront), and
// with more than 128 value columns in long prompts only.  Prompts of 2048 through three such layers of width 1024, time with 32 over with 16: heads of 64 x 64, 16 and 128 of them,
// 0.87 and 0.93; 128 x 64, 32: 0.92; 128 x 128, 64 and 128: 0.985 and 1.055; 256 x 64, 16: 0.89; 192 x 192, 16 and 48: 0.99 (700 positions 1.06) and 1.05;
// 256 x 128, 32: 1.04; 256 x 256, 4, 8, 16 and 64: 0.60, 0.91, 1.03 and 1.13; 128 x 256, 16 and 64: 0.95 and 1.10; 64 x 256, 32 and 96: 1.00 and 1.05.  Of 300 and 64
// positions, 64 x 256, 32: 1.08 and 1.04; 256 x 256, 8: 1.01 and 1.08; 128 x 256, 16: 1.00 and 1.04; 128 x 64, 32: 1.00 and 0.99.
#define DELTA_WIDE_M 512
inline bool delta_wide_chunks(const DeltaShape &d, int M) {
    const DeltaRec r = delta_rec(d);
    return (int64_t)d.H * 256 * r.NT * r.NC <= (d.D > 128 ? 2 : 3) << 18 && (d.V <= 128 || M >= DELTA_WIDE_M);
}

// the longest prompt, of up to M tokens, that goes in chunks of 16 (0: none)
inline int delta_most16(const DeltaShape &d, int M) {
    if (M < L_DELTA_WALK_MIN) return 0;
    if (!delta_wide_chunks(d, M)) return M;
    return delta_wide_chunks(d, L_DELTA_WALK_MIN) ? 0 : std::min(M, DELTA_WIDE_M - 1);
}

// Chunks of 32 a pass, passes of about the same length.  A record holds a state, so that those of a whole prompt are 1.9 times (heads of 128 x 128) what chunks of 16
// and their outputs take: 138 MB for 2048 positions of 16 heads.  With 160 MiB that is one pass; 32 heads have two, which is as fast as one (3.37 and 3.41 ms through
// three layers of width 4096: the records then stay in the memory-side cache).  Smaller passes cost: 16 heads 1.65 ms in one, 1.67 in two, 1.77 in three, 1.90 in five.
#define DELTA_RECORDS ((int64_t)40 << 20)  // floats
#define DELTA_LEAST_CHUNKS 8               // ... or as many chunks
inline int delta_pass_chunks(const DeltaShape &d, int M, int64_t floats) {
    const int n = (M + WK_T - 1) / WK_T;
    const int64_t most = floats / delta_chunk_floats(d), passes = most < 1 ? 0 : (n + most - 1) / most;
    return passes ? (int)((n + passes - 1) / passes) : 0;
}
// scratch for prompts of up to M tokens, and what there has to be of it
struct DeltaScratch {
    int64_t floats, least;
};
inline DeltaScratch delta_walk_scratch(const DeltaShape &d, int M) {
    DeltaScratch s{0, 0};
    const int64_t chunk = delta_chunk_floats(d);
    if (delta_wide_chunks(d, M)) {
        s.floats = std::min<int64_t>((M + WK_T - 1) / WK_T, std::max<int64_t>(DELTA_LEAST_CHUNKS, DELTA_RECORDS / chunk)) * chunk;
        s.least = chunk;
    }
    const int most16 = delta_most16(d, M);
    s.least = std::max(s.least, delta_rec16_floats(d, most16));
    s.floats = std::max(s.floats, s.least);
    return s;
}
// What there is of it then, `have` before: memory of s.floats or, where that is not to be had, of less, down to what there has to be (0: not even that).
// get(n) says whether it got n floats.
template <class F>
inline int64_t delta_scratch_get(const DeltaScratch &s, int64_t have, F get) {
    for (int64_t n = s.floats; n > have; n = std::max(s.least, n / 2)) {
        if (get(n)) return n;
        if (n <= s.least) break;
    }
    return have >= s.least ? have : 0;
}
// rows of outputs that the walk in chunks of 16 or the scan leaves for the head norm, for prompts of up to M tokens
inline int delta_out_rows(const DeltaShape &d, int M) { return (std::max(delta_most16(d, M), std::min(M, L_DELTA_WALK_MIN - 1)) + 15) / 16 * 16; }
