// The products of k_gemm.hip for few positions, few rows, or both: C[m][n] = sum_k X[m][k] W[n][k] where tiles of 64 x 64 results
// would leave most of the chip without one.
//
// What bounds such a product is reading the matrix once, so as many wavefronts as possible have a share of it under way.
//
// few_kernel (fp32, and bf16 of up to 16 positions or few inputs): a workgroup takes 16 or 32 rows and 16 to 64 positions, its eight wavefronts an eighth of the inputs each, and
// their sums are added in LDS, in order.  Operands go from memory straight to the registers that the matrix instructions take (a lane holds 8 consecutive
// inputs of one row), the next step's under way during this one's; a position's inputs come from the L2.  A load's 16 rows lie a multiple of 4 KB apart, which
// is what bounds it from 17 positions on.
//
// few_ring_kernel (bf16, few_ring.h): whole lines, through LDS.  Microseconds of few_kernel and of this, a matrix of its own in each launch: 64 positions,
// 16 384 rows x 2048 inputs 30.6, 17.1; 28 672 x 4096 106, 49.9; 4096 x 14 336 81.7, 30.4; 2048 x 8192 24.7, 13.5; 3072 x 2048 14.3, 8.2; a router's 32 rows x 4096, 12.6, 5.3; 16 experts of 2048 x 2048, 14 and 64 positions each: 43, 28.6 and 124, 47.8.
#include "few_ring.h"
#include "layered_gemm.h"

typedef __bf16 few_bf16x8 __attribute__((ext_vector_type(8)));
typedef float few_f32x4 __attribute__((ext_vector_type(4)));

#define FEW_WAVES 8

// one step's operands of a lane: UK groups of 32 inputs
template <int PREC, int RN, int JM, int UK>
struct FewStep {
    uint4 w[RN][UK];
    uint4 x[JM][UK][PREC ? 2 : 1];
};

// rows n0 .. n0 + 16 RN - 1 of W, positions m0 .. m0 + 16 JM - 1 of a block of mcount that starts at row mb
template <int PREC, int EPI, int RN, int JM>
__device__ __forceinline__ void few_item(const GemmArgs &a, const uint16_t *W, int64_t n0, int64_t mb, int m0, int mcount, float *s_red) {
    constexpr int UK = RN * JM * (1 + PREC) > 4 ? 1 : 2, TN = 16 * RN, TM = 16 * JM, NQ = TN / 4;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int units = a.ld / (32 * UK), u0 = units * wave / FEW_WAVES, u1 = units * (wave + 1) / FEW_WAVES;  // (ld is a multiple of 64)
    const int at = 8 * (lane >> 4);
    const uint16_t *wp[RN];
    const char *xp[JM];
#pragma unroll
    for (int i = 0; i < RN; i++) wp[i] = W + min(n0 + 16 * i + (lane & 15), a.n_rows - 1) * a.ld + at;
#pragma unroll
    for (int j = 0; j < JM; j++) {
        int64_t row = mb + min(m0 + 16 * j + (lane & 15), mcount - 1);  // (rows past the end repeat the last one; not stored)
        if (a.gather) row = a.gather[row];
        xp[j] = (const char *)a.x + (row * a.ldx + at) * (PREC ? 4 : 2);
    }
    auto fetch = [&](FewStep<PREC, RN, JM, UK> &f, int step) {
        const int k = step * 32 * UK;
#pragma unroll
        for (int u = 0; u < UK; u++) {
#pragma unroll
            for (int i = 0; i < RN; i++) f.w[i][u] = *(const uint4 *)(wp[i] + k + 32 * u);
#pragma unroll
            for (int j = 0; j < JM; j++)
#pragma unroll
                for (int p = 0; p < (PREC ? 2 : 1); p++) f.x[j][u][p] = *(const uint4 *)(xp[j] + (k + 32 * u) * (PREC ? 4 : 2) + 16 * p);
        }
    };
    few_f32x4 acc[RN][JM];
#pragma unroll
    for (int i = 0; i < RN; i++)
#pragma unroll
        for (int j = 0; j < JM; j++) acc[i][j] = few_f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const FewStep<PREC, RN, JM, UK> &f) {
#pragma unroll
        for (int u = 0; u < UK; u++) {
            if constexpr (PREC == 0) {
#pragma unroll
                for (int i = 0; i < RN; i++)
#pragma unroll
                    for (int j = 0; j < JM; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(few_bf16x8, f.w[i][u]),
                                                                            __builtin_bit_cast(few_bf16x8, f.x[j][u][0]), acc[i][j], 0, 0, 0);
            } else {
                // (instruction e contracts the inputs 8 (lane / 16) + e of both operands)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    float A[RN], B[JM];
#pragma unroll
                    for (int i = 0; i < RN; i++) {
                        const uint32_t w = e < 2 ? f.w[i][u].x : e < 4 ? f.w[i][u].y : e < 6 ? f.w[i][u].z : f.w[i][u].w;
                        A[i] = e & 1 ? l_bf16_hi(w) : l_bf16_lo(w);
                    }
#pragma unroll
                    for (int j = 0; j < JM; j++) {
                        const uint4 x = f.x[j][u][PREC ? e >> 2 : 0];
                        B[j] = __uint_as_float((e & 3) == 0 ? x.x : (e & 3) == 1 ? x.y : (e & 3) == 2 ? x.z : x.w);
                    }
#pragma unroll
                    for (int i = 0; i < RN; i++)
#pragma unroll
                        for (int j = 0; j < JM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[i], B[j], acc[i][j], 0, 0, 0);
                }
            }
        }
    };
    if (u0 < u1) {
        FewStep<PREC, RN, JM, UK> cur, nxt;
        fetch(cur, u0);
        for (int u = u0; u + 1 < u1; u++) {
            fetch(nxt, u + 1);
            multiply(cur);
            cur = nxt;
        }
        multiply(cur);
    }
    // sums [wavefront][position][quad of rows], a position's quads turned by the position: 16 lanes write 16 different slots
#pragma unroll
    for (int i = 0; i < RN; i++)
#pragma unroll
        for (int j = 0; j < JM; j++) {
            const int p = 16 * j + (lane & 15), q = (4 * i + (lane >> 4)) ^ (p & (NQ - 1));
            *(few_f32x4 *)(s_red + 4 * ((wave * TM + p) * NQ + q)) = acc[i][j];
        }
    __syncthreads();
    for (int o = t; o < TM * NQ; o += 64 * FEW_WAVES) {
        const int p = o / NQ, q = o % NQ;
        few_f32x4 v = *(few_f32x4 *)(s_red + 4 * (p * NQ + (q ^ (p & (NQ - 1)))));
#pragma unroll
        for (int w = 1; w < FEW_WAVES; w++) v += *(few_f32x4 *)(s_red + 4 * ((w * TM + p) * NQ + (q ^ (p & (NQ - 1)))));
        if (m0 + p < mcount)
            gemm_store4<PREC, EPI>(a, mb + m0 + p, n0 + 4 * q, gemm_row<EPI>(a, mb + m0 + p), gemm_col<EPI>(a, n0 + 4 * q), v.x, v.y, v.z, v.w);
    }
}

// bf16, rows n0 .. n0 + TN - 1 of W x positions m0 .. m0 + TM - 1; store(quads of the tile, sum) takes the sums of steps k0 .. k1 of 64 inputs
template <int TN, int TM, class Store>
__device__ __forceinline__ void few_ring_sums(const GemmArgs &a, const uint16_t *W, int64_t n0, int64_t mb, int m0, int mcount, int k0, int k1, unsigned char *s,
                                              Store store) {
    constexpr int LA = TN / 8, LX = TM / 8;
    const int t = threadIdx.x, lane = t & 63;
    const uint16_t *wp[LA], *xp[LX];
#pragma unroll
    for (int i = 0; i < LA; i++) wp[i] = W + min(n0 + few_ring_row(i, lane), a.n_rows - 1) * a.ld + 64 * k0 + 8 * few_ring_chunk(i, lane);
#pragma unroll
    for (int i = 0; i < LX; i++) {
        int64_t row = mb + min(m0 + few_ring_row(i, lane), mcount - 1);  // (rows past the end repeat the last one; not stored)
        if (a.gather) row = a.gather[row];
        xp[i] = (const uint16_t *)a.x + row * a.ldx + 64 * k0 + 8 * few_ring_chunk(i, lane);
    }
    few_ring<TN, TM, FewQuarters>(k1 - k0, blockIdx.x >> 3, s, [&](int i, int k) { return wp[i] + 64 * k; }, [&](int i, int k) { return xp[i] + 64 * k; });
    for (int o = t; o < TM * TN / 4; o += 256) store(o, few_ring_sum<TN, TM>(s, o / (TN / 4), o % (TN / 4)));
}
template <int EPI, int TN>
__device__ __forceinline__ void few_ring_store(const GemmArgs &a, int64_t n0, int64_t mb, int m0, int mcount, int o, float4 v) {
    const int p = o / (TN / 4);
    const int64_t n = n0 + 4 * (o % (TN / 4));
    if (m0 + p < mcount) gemm_store4<0, EPI>(a, mb + m0 + p, n, gemm_row<EPI>(a, mb + m0 + p), gemm_col<EPI>(a, n), v.x, v.y, v.z, v.w);
}
// `splits` workgroups share an item's inputs.  Each leaves its sums in a.part; the one that is through last (a.arrived: zero between launches) adds all of them,
// in order, so that nobody waits.
template <int EPI, int TN, int TM>
__global__ __launch_bounds__(256) void few_ring_kernel(GemmArgs a, unsigned n_nt, unsigned n_mt, unsigned splits) {
    extern __shared__ __align__(16) unsigned char s_ring[];
    __shared__ unsigned s_before;
    const unsigned n_items = n_nt * n_mt * splits, per = (n_items + 7) / 8, k = blockIdx.x >> 3, id = (blockIdx.x & 7u) * per + k;
    if (k >= per || id >= n_items) return;
    const unsigned item = id / splits, part = id % splits;
    const int64_t n0 = (int64_t)(item / n_mt) * TN;
    const int m0 = (int)(item % n_mt) * TM, nk = a.ld >> 6, t = threadIdx.x;
    if (splits == 1) {
        few_ring_sums<TN, TM>(a, a.w, n0, 0, m0, a.M, 0, nk, s_ring, [&](int o, float4 v) { few_ring_store<EPI, TN>(a, n0, 0, m0, a.M, o, v); });
        return;
    }
    typedef unsigned long long u64;
    constexpr int QUADS = TM * TN / 4;
    u64 *mine = (u64 *)(a.part + (int64_t)id * 4 * QUADS);
    few_ring_sums<TN, TM>(a, a.w, n0, 0, m0, a.M, (int)(nk * part / splits), (int)(nk * (part + 1) / splits), s_ring, [&](int o, float4 v) {
        // (halves of a quad apart, so that lanes store consecutive words)
        __hip_atomic_store(mine + o, (u64)__float_as_uint(v.x) | (u64)__float_as_uint(v.y) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(mine + QUADS + o, (u64)__float_as_uint(v.z) | (u64)__float_as_uint(v.w) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    });
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the sums have been written where everyone reads them
    __syncthreads();
    if (t == 0) {
        s_before = __hip_atomic_fetch_add(a.arrived + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (s_before == splits - 1) __hip_atomic_store(a.arrived + item, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (s_before != splits - 1) return;
    const u64 *all = (const u64 *)(a.part + (int64_t)item * splits * 4 * QUADS);
    for (int o = t; o < QUADS; o += 256) {
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
        for (unsigned p = 0; p < splits; p++) {
            const u64 lo = __hip_atomic_load(all + 2 * QUADS * p + o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const u64 hi = __hip_atomic_load(all + 2 * QUADS * p + QUADS + o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            v.x += __uint_as_float((unsigned)lo);
            v.y += __uint_as_float((unsigned)(lo >> 32));
            v.z += __uint_as_float((unsigned)hi);
            v.w += __uint_as_float((unsigned)(hi >> 32));
        }
        few_ring_store<EPI, TN>(a, n0, 0, m0, a.M, o, v);
    }
}
// an expert's rows, 64 positions at a time or what is left
template <int EPI, int TN>
__global__ __launch_bounds__(256) void few_ring_grouped_kernel(GemmArgs a, unsigned n_nt) {
    extern __shared__ __align__(16) unsigned char s_ring[];
    const unsigned n_items = (unsigned)a.n_tiles[0] * n_nt, per = (n_items + 7) / 8, k = blockIdx.x >> 3, item = (blockIdx.x & 7u) * per + k;
    if (k >= per || item >= n_items) return;
    const GemmTile g = a.tiles[item / n_nt];
    const uint16_t *w = a.w + g.expert * a.expert_stride;
    const int64_t n0 = (int64_t)(item % n_nt) * TN;
    for (int m0 = 0; m0 < g.n; m0 += 64) {
        if (m0) __syncthreads();
        auto store = [&](int o, float4 v) { few_ring_store<EPI, TN>(a, n0, g.row0, m0, g.n, o, v); };
        if (g.n - m0 <= 32)
            few_ring_sums<TN, 32>(a, w, n0, g.row0, m0, g.n, 0, a.ld >> 6, s_ring, store);
        else
            few_ring_sums<TN, 64>(a, w, n0, g.row0, m0, g.n, 0, a.ld >> 6, s_ring, store);
    }
}

// Items (rows, positions) are dealt to the 8 XCDs as contiguous runs, positions fastest: workgroups on the same rows share an L2.
template <int PREC, int EPI, int RN, int JM>
__global__ __launch_bounds__(64 * FEW_WAVES) void few_kernel(GemmArgs a, unsigned n_nt, unsigned n_mt) {
    __shared__ __align__(16) float s_red[FEW_WAVES * 16 * JM * 16 * RN];
    const unsigned n_items = n_nt * n_mt, per = (n_items + 7) / 8, k = blockIdx.x >> 3, item = (blockIdx.x & 7u) * per + k;
    if (k >= per || item >= n_items) return;
    few_item<PREC, EPI, RN, JM>(a, a.w, (int64_t)(item / n_mt) * 16 * RN, 0, (int)(item % n_mt) * 16 * JM, a.M, s_red);
}

// an expert's rows: as many positions at a time as it was chosen for
template <int PREC, int EPI>
__global__ __launch_bounds__(64 * FEW_WAVES) void few_grouped_kernel(GemmArgs a, unsigned n_nt) {
    __shared__ __align__(16) float s_red[FEW_WAVES * 64 * 16];
    const unsigned n_items = (unsigned)a.n_tiles[0] * n_nt, per = (n_items + 7) / 8, k = blockIdx.x >> 3, item = (blockIdx.x & 7u) * per + k;
    if (k >= per || item >= n_items) return;
    const GemmTile g = a.tiles[item / n_nt];
    const uint16_t *w = a.w + g.expert * a.expert_stride;
    const int64_t n0 = (int64_t)(item % n_nt) * 16;
    if (g.n <= 16) {
        few_item<PREC, EPI, 1, 1>(a, w, n0, g.row0, 0, g.n, s_red);
    } else if (g.n <= 32) {
        few_item<PREC, EPI, 1, 2>(a, w, n0, g.row0, 0, g.n, s_red);
    } else {
        for (int m0 = 0; m0 < g.n; m0 += 64) {
            if (m0) __syncthreads();
            few_item<PREC, EPI, 1, 4>(a, w, n0, g.row0, m0, g.n, s_red);
        }
    }
}

// ---- which kernel, for bf16 ----
// us, few_kernel, then tiles of 32 x 32, 64 x 32, 32 x 64 and 64 x 64 results (rows x positions); S: workgroups that share a tile's inputs
//   3072 x 2048,  24 positions:  7.7 |  7.4,  9.5,  8.7, 12.1      16 384 x 2048, 32: 26.8 | 17.0, 15.0, 18.0, 15.6
//                 64:           14.3 |  8.2,  9.8,  9.4, 13.0                     64: 30.6 | 27.1, 21.8, 20.7, 17.1
//                128:           19.6 | 12.6, 10.4,  9.9, 12.8      28 672 x 4096, 32: 85.2 | 50.2, 42.8, 54.1, 44.5
//                192:           26.1 | 15.5, 13.5, 15.4, 11.9                     64: 106  | 76.7, 64.8, 61.9, 49.9
//   2048 x 8192,  32: 24.7 | 20.3 S1, 11.1 S4; 64: 24.7 | 16.0 S2 in 32 x 32, 25.5 S1, 13.5 S4 in 32 x 64
//   4096 x 14 336, 32: 42.2 | 38.1 S1, 26.3 S2; 64: 81.7 | 32.7 S2 in 32 x 64, 30.4 S4 in 64 x 64
//   32 x 4096, 64: 12.6 | 6.9 S1, 5.3 S4; 2048 x 2048, 24: 7.6 | 7.0 S1, 7.3 S2 (a share costs 1.7 us, and a step of 64 inputs 0.05 to 0.1)
// So: the smallest tiles that come to at most one a compute unit (of many inputs, where they can be shared out, all positions up to 64 in one tile), and the
// largest beyond.  Up to 16 positions few_kernel's 16 x 16 results have more workgroups: 2 to 16 positions of 2048 x 2048 5.5 to 6.5 | 6.0 to 6.6, 4096 x 4096 9.2 to
// 10.3 | 10.4 to 10.6, but 2048 x 8192 13.8 to 17.1 | 10.5 to 10.8 S4, 4096 x 14 336 24.6 to 28.8 | 23.9 to 24.2 S2, 8 of 16 384 x 2048 15.3 | 14.4.
//
// All of that is of many inputs.  A tile of the ring costs the fill of its LDS and its epilogue, which nothing hides (one workgroup a compute unit), so with fewer inputs, in steps of 64,
// it has to be one of a full round.  The ring's time over few_kernel's, worst of four epilogues:
//   one round: 8 steps and more 0.5 to 1.04.  4 (256 inputs): 2048 rows, 24 to 128 positions 0.85 to 1.02; 4096, 17 and 64 1.06 and 0.86; 8192, 17 and 64 (tiles of 64 rows) 0.98 and
//     1.00; 8192 and 16 384, 128 and 33 1.10 and 1.16.  6: 4096, 17 1.03, 64 0.81; 8192, 128 0.97; 16 384, 33 1.05.  Below 4, 17 to 128 positions 0.9 to 1.8.
//   more: 4 to 7 steps 1.0 to 1.4 (32 000 rows, 32 positions 0.96 to 1.04).  8: 16 384 rows, 32 positions 0.90; 20 480 1.14, 28 672 0.97; 33 of 28 672 1.05, 64 0.99.  12: 18 432, 17, 32 and 64
//     1.19, 1.01 and 0.99; 28 672, 17 0.94.  16: 18 432, 17 and 24 1.10 and 0.98; 24 576, 17 0.97.  24: 18 432, 17 0.99.  From 65 positions on of 12 and more 0.6 to 1.02.
//   up to 16 positions: 12: 16 384, 5 and 16 1.06 and 0.93.  32: 16 384 rows, 5, 8 and 16 positions 1.01, 0.95 and 0.78; 20 480 1.25, 1.13 and 0.99; 28 672 1.07, 0.97 and 0.82.  64: 1.0, 0.9 and 0.7; 1.12,
//     1.0 and 0.87; 0.95, 0.85 and 0.70.
// Steps times the results' share of the rounds' room, against 6.5, is the line that those lie on two sides of.
struct FewPlan {
    int rows = 0, positions = 0;  // of a tile (0: few_kernel)
    unsigned splits = 1;
};
static FewPlan few_plan(const GemmArgs &a, int64_t cols) {
    FewPlan p;
    const int nk = a.ld / 64;
    if (nk < 4) return p;
    auto tiles = [&](int rows, int positions) { return (cols + rows - 1) / rows * ((a.M + positions - 1) / positions); };
    if (tiles(32, 32) <= FEW_PART_ITEMS && (a.M <= 32 || nk < 64))
        p.rows = p.positions = 32;
    else if (a.M > 32 && tiles(32, 64) <= FEW_PART_ITEMS && !(nk >= 128 && a.M <= 64 && tiles(32, 64) > 64))
        p.rows = 32, p.positions = 64;
    else
        p.rows = 64, p.positions = a.M <= 32 ? 32 : 64;
    const int64_t n = tiles(p.rows, p.positions), rounds = (n + FEW_PART_ITEMS - 1) / FEW_PART_ITEMS;
    if (nk >= 64 && a.part && a.arrived) p.splits = (unsigned)max((int64_t)1, min((int64_t)min(8, nk / 16), FEW_PART_ITEMS / n));
    const bool filled = 2 * nk * cols * a.M >= 13 * rounds * FEW_PART_ITEMS * p.rows * p.positions;
    bool ring;
    if (a.M <= 16)
        ring = p.splits >= 4 || (p.splits >= 2 && nk >= 128) || (n >= FEW_PART_ITEMS && filled);
    else if (rounds == 1)
        ring = nk >= 8 || (!(nk < 6 && p.rows == 64) && (a.M > 32 || n > FEW_PART_ITEMS / 2));
    else
        ring = nk >= 8 && (filled || a.M > 64);
    if (!ring) p.rows = 0;
    return p;
}
template <int EPI, int TN, int TM>
static hipError_t few_ring_plain(hipStream_t s, const GemmArgs &a, int64_t cols, unsigned splits) {
    static bool set[FEW_RING_DEVICES] = {};
    const unsigned n_nt = (unsigned)((cols + TN - 1) / TN), n_mt = (unsigned)((a.M + TM - 1) / TM);
    return few_ring_go(s, few_ring_kernel<EPI, TN, TM>, set, few_ring_lds(TN, TM), (int64_t)n_nt * n_mt * splits, a, n_nt, n_mt, splits);
}
template <int EPI, int TN>
static hipError_t few_ring_grouped(hipStream_t s, const GemmArgs &a, int64_t cols) {
    static bool set[FEW_RING_DEVICES] = {};
    const unsigned n_nt = (unsigned)((cols + TN - 1) / TN);
    return few_ring_go(s, few_ring_grouped_kernel<EPI, TN>, set, max(few_ring_lds(TN, 32), few_ring_lds(TN, 64)), (int64_t)a.max_tiles * n_nt, a, n_nt);
}
template <int PREC, int EPI>
static hipError_t few_launch(hipStream_t s, const GemmArgs &a, int64_t cols) {
    if (a.tiles) {
        if constexpr (EPI == GE_STORE || EPI == GE_UP || EPI == GE_GLU) {
            if constexpr (PREC == 0) {
                // us, few_grouped_kernel and tiles of 32 and 64 rows; 8 matrices of 512 x 512 (64 tiles of 64 rows), 8, 16 and 48 positions each: 3.6, 4.0, 6.5;
                // 3.9, 4.0, 6.1; 4.6, 4.8, 7.9; of 2048 x 1024 (256): 11.0, 13.8, 30.4; 11.1, 11.6, 17.8; 9.5, 9.9, 15.0; 16 of 2048 x 2048, 2, 16 and 64 each:
                // 29.2, 42.9, 124; 27.6, 29.9, 53.9; 27.8, 28.6, 47.8.
                // So: 64 rows where that gives most compute units a tile, and as many to each (250 tiles 0.8 to 1.02 of few_grouped_kernel's time, 280 to 340 1.0 to 1.3; of 64 to 192 inputs and
                // 48 positions each 1.0 to 1.2 with a gate), otherwise 32 rows where the loop is long enough for the fill of the ring and its epilogue.  Their time over
                // few_grouped_kernel's, 32 to 128 tiles of 64 rows, 9, 16, 32 and 48 positions each, stored: 256 inputs 1.1, 1.05, 1.0 to 1.1, 0.9 to 1.0; 512 1.05, 0.95, 0.8 to 1.0, 0.7
                // to 0.9; 2048 1.0 to 1.1, 0.75 to 1.0, 0.6 to 0.9, 0.5 to 0.8; with a gate: 512 1.04 to 1.14, 1.0 to 1.1, 1.02 to 1.3, 0.94 to 1.2; 2048 1.1, 0.95 to 1.1, 0.9 to 1.2, 0.7 to 1.06,
                // the smaller figures at 128 tiles.
                const int64_t nk = a.ld / 64, each = a.rows_each, wide = few_blocks(a, cols), rounds = (wide + FEW_PART_ITEMS - 1) / FEW_PART_ITEMS;
                constexpr bool stored = EPI == GE_STORE;
                if (3 * wide >= 2 * FEW_PART_ITEMS * rounds) {
                    if (nk >= 4 || each <= 32 || (stored && nk >= 2)) return few_ring_grouped<EPI, 64>(s, a, cols);
                } else if (stored ? nk >= 6 && nk * each >= 160 : (wide >= 80 && nk * each >= 384) || nk * each >= 1600) {
                    return few_ring_grouped<EPI, 32>(s, a, cols);
                }
            }
            const unsigned n_nt = (unsigned)((cols + 15) / 16), most = (unsigned)a.max_tiles * n_nt;
            hipLaunchKernelGGL((few_grouped_kernel<PREC, EPI>), dim3(8 * ((most + 7) / 8)), dim3(64 * FEW_WAVES), 0, s, a, n_nt);
            return hipGetLastError();
        }
        return hipErrorInvalidValue;
    }
    if constexpr (PREC == 0) {
        const FewPlan p = few_plan(a, cols);
        if (p.rows == 32) return p.positions == 32 ? few_ring_plain<EPI, 32, 32>(s, a, cols, p.splits) : few_ring_plain<EPI, 32, 64>(s, a, cols, p.splits);
        if (p.rows == 64) return p.positions == 32 ? few_ring_plain<EPI, 64, 32>(s, a, cols, p.splits) : few_ring_plain<EPI, 64, 64>(s, a, cols, p.splits);
    }
#define GO(RN, JM)                                                                                                                        \
    do {                                                                                                                                  \
        const unsigned n_nt = (unsigned)((cols + 16 * RN - 1) / (16 * RN)), n_mt = (unsigned)((a.M + 16 * JM - 1) / (16 * JM));          \
        hipLaunchKernelGGL((few_kernel<PREC, EPI, RN, JM>), dim3(8 * ((n_nt * n_mt + 7) / 8)), dim3(64 * FEW_WAVES), 0, s, a, n_nt, n_mt); \
        return hipGetLastError();                                                                                                         \
    } while (0)
    if (a.M <= 16) GO(1, 1);
    // 32 rows and 64 positions at a time where that gives every CU a workgroup: half the reads of the positions (fp32 products of that size go to k_gemm's tiles)
    if constexpr (PREC == 0)
        if (a.M > 32 && ((cols + 31) / 32) * ((a.M + 63) / 64) >= 256) GO(2, 4);
    GO(1, 2);
#undef GO
}

hipError_t k_few(hipStream_t s, const GemmArgs &a, int prec, int epi, int64_t cols) {
#define GO(E) \
    case E: return prec ? few_launch<1, E>(s, a, cols) : few_launch<0, E>(s, a, cols)
    switch (epi) {
        GO(GE_STORE);
        GO(GE_RESID);
        GO(GE_ACT);
        GO(GE_UP);
        GO(GE_EMBED);
        GO(GE_DECAY);
        GO(GE_SIGMOID);
        GO(GE_GLU);
    }
#undef GO
    return hipErrorInvalidValue;
}
