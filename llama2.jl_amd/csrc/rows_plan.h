// How k_rows.hip deals out a matrix: workgroups, and the LDS of one.
#pragma once

#include <algorithm>

#include "layered.h"

#define ROWS_THREADS 512
#define ROWS_WAVES 8
#define ROWS_MAX_PAIRS 4096  // row pairs of a workgroup at most: 32 KB of results
#define ROWS_LDS (152 * 1024)

inline int rows_vectors(const RowsArgs &a, int pro) { return pro == RP_DOWN ? a.top : 1; }

// LDS of a workgroup of `pairs` row pairs: the vectors, then the results, where the choice of experts has its logits before
inline size_t rows_lds(const RowsArgs &a, int pro, int64_t pairs) {
    return ((size_t)rows_vectors(a, pro) * a.ld + std::max<size_t>(2 * (size_t)pairs, pro == RP_UP ? a.n_experts : 0)) * sizeof(float);
}

// steps of 512 u inputs (rows_kernel) in all
inline int64_t rows_steps(const RowsArgs &a, int pro, int u) {
    return (a.n_rows + 1) / 2 * rows_vectors(a, pro) * ((a.ld + 512 * u - 1) / (512 * u));
}

// LDS of a workgroup beside rows_lds(), rounded up: sums, and behind a choice of experts each wavefront's own (2464 bytes; 352 and fewer otherwise)
inline size_t rows_fixed_lds(int pro) { return (pro == RP_UP ? 3 : 2) * 1024; }

// two workgroups per CU where LDS holds their vectors and results
inline int64_t rows_most(const RowsArgs &a, int pro, int n_cu) {
    const int64_t pairs = (a.n_rows + 1) / 2;
    const size_t lds = rows_lds(a, pro, std::min<int64_t>(ROWS_MAX_PAIRS, pairs / (2 * n_cu) + 1)) + rows_fixed_lds(pro);
    return (lds > 80 * 1024 ? 1 : 2) * (int64_t)n_cu;
}

// workgroups: no more than that while there is a step for every wavefront and, beside the vectors, LDS for the results
// (32 768 inputs leave room for 3072 pairs)
inline int64_t rows_grid(const RowsArgs &a, int pro, int n_cu, int u) {
    const int64_t pairs = (a.n_rows + 1) / 2, vectors = (int64_t)rows_vectors(a, pro) * a.ld;
    const int64_t room = std::max<int64_t>(2, std::min<int64_t>(ROWS_MAX_PAIRS, (ROWS_LDS / 4 - vectors) / 2));
    const int64_t n = std::max<int64_t>(1, std::min(std::min(rows_most(a, pro, n_cu), pairs), (rows_steps(a, pro, u) + ROWS_WAVES - 1) / ROWS_WAVES));
    return std::max(n, (pairs + room - 2) / (room - 1));
}

// n / d for n < 2^31 by a product and a shift (mul = ceil(2^(32 + shift) / d), 2^shift <= d < 2^(shift + 1): n (mul d - 2^(32 + shift)) < n d <
// 2^(32 + shift)).  What a wavefront loads first lies behind such divisions, and the compiler's way, through floats and back to the scalar unit, takes
// 0.1 us of a launch of 3.
struct RowsDiv {
    unsigned mul, shift, one;  // one: d is 1
};
inline RowsDiv rows_div(unsigned d) {
    if (d <= 1) return {0u, 0u, 1u};
    unsigned s = 0;
    while (d >> (s + 1)) s++;
    if (d == 1u << s) return {0x80000000u, s - 1, 0u};
    return {(unsigned)((((unsigned long long)1 << (32 + s)) + d - 1) / d), s, 0u};
}
__host__ __device__ inline unsigned rows_quot(unsigned n, const RowsDiv &v) {
    const unsigned q = (unsigned)((unsigned long long)n * v.mul >> 32) >> v.shift;
    return v.one ? n : q;
}

// how a matrix's rows are dealt out: workgroup b has `pairs` row pairs, and one more for b < more, one after another
struct RowsPlan {
    int plane;              // half of a staged vector's floats
    int pairs, more;
    int per_vec, per_pair;  // steps of a row pair per staged vector, in all
    RowsDiv by_vec, by_pair, by_each;  // (of rows_each)
    float inv_K;
};
inline RowsPlan rows_plan(const RowsArgs &a, int pro, int u, int64_t grid) {
    const int64_t pairs = (a.n_rows + 1) / 2;
    RowsPlan pl;
    pl.plane = a.ld / 2;
    pl.pairs = (int)(pairs / grid);
    pl.more = (int)(pairs % grid);
    pl.per_vec = (a.ld + 512 * u - 1) / (512 * u);
    pl.per_pair = rows_vectors(a, pro) * pl.per_vec;
    pl.by_vec = rows_div((unsigned)pl.per_vec);
    pl.by_pair = rows_div((unsigned)pl.per_pair);
    pl.by_each = rows_div((unsigned)std::max<int64_t>(1, a.rows_each));
    pl.inv_K = 1.0f / (float)a.K;
    return pl;
}
