// Many tokens through a bf16 matrix, C[m][n] = sum_k X[m][k] W[n][k], on the matrix cores: bf16 activations, or fp32
// ones in three bf16 parts (v_mfma_f32_32x32x16_bf16, fp32 sums), with fused epilogues and a grouped
// form for mixtures of experts; and the row-wise kernels around the products.
#include "layered_gemm.h"

typedef __bf16 l_bf16x8 __attribute__((ext_vector_type(8)));
typedef float l_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t l_u32x4 __attribute__((ext_vector_type(4)));

// Placement of the 16-byte chunks of a 128-byte tile row: 16 consecutive rows' chunks of one index fall into different slots
// of the 256-byte bank row.
__device__ __forceinline__ int gemm_swz(int r) { return (r >> 1) & 7; }

template <int EPI, int TN, int TM, bool GROUPED>
__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs a) {
    constexpr int IN = TN / 64, JM = TM / 64;  // 32 x 32 tiles per wavefront (2 x 2 wavefronts)
    constexpr int KSTEP = 64, OPERANDS = (TN + TM) * 128, RESULTS = 4 * 4 * gemm_epilogue_floats(IN, JM);
    __shared__ __align__(16) unsigned char s_raw[OPERANDS > RESULTS ? OPERANDS : RESULTS];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wn = wave & 1, wm = wave >> 1;
    const uint16_t *W = a.w;
    int64_t mb = 0;
    int mcount = a.M;
    const int64_t n0 = (int64_t)blockIdx.y * TN;
    int m0 = blockIdx.x * TM;
    if (GROUPED) {
        if ((int)blockIdx.x >= a.n_tiles[0]) return;
        const GemmTile gt = a.tiles[blockIdx.x];
        W += gt.expert * a.expert_stride;
        mb = gt.row0;
        mcount = gt.n;
        m0 = 0;
    }
    l_f32x16 acc[IN][JM];
#pragma unroll
    for (int i = 0; i < IN; i++)
#pragma unroll
        for (int j = 0; j < JM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    // rows this thread copies: row t / 8 + 32 i of each tile, elements 8 (t % 8) .. of a step
    constexpr int WL = TN / 32, XL = TM / 32;
    const int c8 = t & 7;
    const uint16_t *wrow[WL], *xrow[XL];
#pragma unroll
    for (int i = 0; i < WL; i++) {
        int64_t r = n0 + (t >> 3) + 32 * i;
        if (r >= a.n_rows) r = a.n_rows - 1;
        wrow[i] = W + r * a.ld + 8 * c8;
    }
#pragma unroll
    for (int i = 0; i < XL; i++) {
        int m = m0 + (t >> 3) + 32 * i;
        if (m >= mcount) m = mcount - 1;  // (repeats the last row; not stored)
        int64_t row = mb + m;
        if (a.gather) row = a.gather[row];
        xrow[i] = (const uint16_t *)a.x + row * a.ldx + 8 * c8;
    }
    // (vectors of the compiler's own: as uint4, a struct, the sixteen words went through scratch memory in every step)
    l_u32x4 wreg[WL], xreg[XL];
    auto gload = [&](int k0) {
#pragma unroll
        for (int i = 0; i < WL; i++) wreg[i] = *(const l_u32x4 *)(wrow[i] + k0);
#pragma unroll
        for (int i = 0; i < XL; i++) xreg[i] = *(const l_u32x4 *)(xrow[i] + k0);
    };
    gload(0);
    for (int k0 = 0; k0 < a.ld; k0 += KSTEP) {
        l_u32x4 *s_w = (l_u32x4 *)s_raw, *s_x = s_w + TN * 8;
#pragma unroll
        for (int i = 0; i < WL; i++) {
            const int r = (t >> 3) + 32 * i;
            s_w[r * 8 + (c8 ^ gemm_swz(r))] = wreg[i];
        }
#pragma unroll
        for (int i = 0; i < XL; i++) {
            const int r = (t >> 3) + 32 * i;
            s_x[r * 8 + (c8 ^ gemm_swz(r))] = xreg[i];
        }
        __syncthreads();
        if (k0 + KSTEP < a.ld) gload(k0 + KSTEP);
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
            const int c = 2 * kk + (lane >> 5);
            l_bf16x8 A[IN], B[JM];
#pragma unroll
            for (int i = 0; i < IN; i++) {
                const int r = (TN / 2) * wn + 32 * i + (lane & 31);
                A[i] = __builtin_bit_cast(l_bf16x8, s_w[r * 8 + (c ^ gemm_swz(r))]);
            }
#pragma unroll
            for (int j = 0; j < JM; j++) {
                const int r = (TM / 2) * wm + 32 * j + (lane & 31);
                B[j] = __builtin_bit_cast(l_bf16x8, s_x[r * 8 + (c ^ gemm_swz(r))]);
            }
#pragma unroll
            for (int i = 0; i < IN; i++)
#pragma unroll
                for (int j = 0; j < JM; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[i], B[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    // (the last barrier of the loop is behind every read of the operands)
    gemm_epilogue<0, EPI, IN, JM>(a, acc, (float *)s_raw + wave * gemm_epilogue_floats(IN, JM), mb, m0 + (TM / 2) * wm, mcount, n0 + (TN / 2) * wn, lane);
}

// eight fp32 values as three bf16 ones each, their sum exactly: the upper eight bits of the 24, the next eight, the last.  (From 2^-110 on: of smaller values the
// last parts are no normal numbers, and what is lost with them is below 2^-126.)
struct GemmParts {
    l_bf16x8 part[3];
};
__device__ __forceinline__ GemmParts gemm_split(float4 a, float4 b) {
    const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t w[3][8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        w[0][e] = __float_as_uint(x[e]);
        const float r = x[e] - __uint_as_float(w[0][e] & 0xFFFF0000u);
        w[1][e] = __float_as_uint(r);
        w[2][e] = __float_as_uint(r - __uint_as_float(w[1][e] & 0xFFFF0000u));
    }
    GemmParts g;
#pragma unroll
    for (int p = 0; p < 3; p++) {
        l_u32x4 u;
#pragma unroll
        for (int q = 0; q < 4; q++) u[q] = __builtin_amdgcn_perm(w[p][2 * q + 1], w[p][2 * q], 0x07060302u);  // (the upper halves of both)
        g.part[p] = __builtin_bit_cast(l_bf16x8, u);
    }
    return g;
}

// fp32 activations, on the bf16 matrix cores, whose rate is sixteen times that of the fp32 ones: weights are bf16, and an activation is the sum of
// three bf16 values (gemm_split), so a product is three of theirs, each exact in the fp32 sums.  Against 64 bits the results are nearer than the
// fp32 instructions' (v_mfma_f32_32x32x2_f32), whose sum takes two products at a time: relative rms error at 256, 1024 and 4096 normal inputs 9.0e-8,
// 1.25e-7 and 1.4e-7, theirs 2.9e-7, 5.8e-7 and 1.2e-6; all positive 5.2e-8, 5.5e-8 and 5.0e-8, theirs 2.5e-7, 4.9e-7 and 9.8e-7.  For that, sums leave the
// matrix cores every FOLD steps: their additions truncate, and 4096 positive inputs in one sum of theirs were 3.2e-6 low.
//
// Tiles of 64 rows and TM positions; a step's operands go through LDS, whole rows of 64 inputs, and each of four wavefronts multiplies a quarter of the step's
// inputs for the whole tile: no operand is read from LDS or split twice.  What bounds a CU is the sum of a step's parts, 48 KB through LDS, 96
// vector instructions to split with and 12 of the matrix cores a wavefront, 0.4 us at 64 positions with two workgroups on the CU.  KS: as many groups of four
// wavefronts in a workgroup, each with a share of the steps: for grids that leave a CU one workgroup.  The fp32 instructions and this, us: 509 positions,
// 4096 x 1024: 41, 20.5; 1024 x 4096: 42, 25; 1608 x 1024: 25, 12.6; 2048 positions, 4096 x 1024: 139, 71; 16 matrices of 2048 x 2048, 64 and 192
// positions each: 132, 43 and 380, 134.  (Activations stored in parts: 6 bytes an element where 4 do, 19 and 39 us for the first two, but products of
// few positions were 1.2 to 1.3 times slower.  Two steps of loads under way: the same.)
// SHORT (for one or two steps; KS 1, TM 64): a wavefront has a quarter of the results instead, over all inputs.  Operands are read from LDS and split twice, but nothing is
// exchanged, which took longer than the products; the sums are the same.  us, tiles of 128 x 128 on the fp32 instructions, otherwise and SHORT: 64 inputs, 16 384 rows with an
// activation, 2048 positions 76, 101, 68; 8192, 300: 10.5, 13.0, 8.6; 128 inputs, 8192 rows, 2048 positions 62, 57, 40; 1024, 300 (3 x 10^5 results) 5.8, 6.7, 6.9.
template <int EPI, bool GROUPED, int KS, int TM, bool SHORT = false>
__global__ __launch_bounds__(256 * KS, 2) void gemm_parts_kernel(GemmArgs a, unsigned n_nt) {
    constexpr int T = 64, KSTEP = 64, BUFFER = (2 * T + 4 * TM) * KSTEP, FOLD = 8, JM = TM / 32, XL = TM / 16;
    extern __shared__ __align__(16) unsigned char s_raw[];  // [KS][2][BUFFER], then the wavefronts' sums
    const int t = threadIdx.x & 255, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const uint16_t *W = a.w;
    int64_t mb = 0;
    int mcount = a.M;
    int64_t n0 = (int64_t)blockIdx.y * T;
    int m0 = blockIdx.x * TM;
    if (GROUPED) {
        // (blockIdx.y: which half of a block.  Items (block, columns) go to the XCDs as contiguous runs, and workgroups without one come last: with those
        // between the others, as the columns of a grid of max_tiles, they fell on the same few CUs, and 8 matrices of 2048 x 2048 took 66 us instead of 31)
        const unsigned n_items = (unsigned)a.n_tiles[0] * n_nt, per = (n_items + 7) / 8, k = blockIdx.x >> 3, item = (blockIdx.x & 7u) * per + k;
        if (k >= per || item >= n_items) return;
        const GemmTile gt = a.tiles[item / n_nt];
        W += gt.expert * a.expert_stride;
        mb = gt.row0;
        mcount = gt.n;
        n0 = (int64_t)(item % n_nt) * T;
        m0 = TM * blockIdx.y;
        if (m0 >= mcount) return;
    }
    // what this thread copies of a step: elements 8 (t % 8) .. of rows t / 8 + 32 i of W, elements 4 (t % 16) .. of rows t / 16 + 16 i of X
    const int steps = a.ld / KSTEP, share = (steps + KS - 1) / KS, first = share * part;
    const uint16_t *wrow[2];
    const float *xrow[XL];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        int64_t r = n0 + (t >> 3) + 32 * i;
        if (r >= a.n_rows) r = a.n_rows - 1;
        wrow[i] = W + r * a.ld + 8 * (t & 7);
    }
#pragma unroll
    for (int i = 0; i < XL; i++) {
        int m = m0 + (t >> 4) + 16 * i;
        if (m >= mcount) m = mcount - 1;  // (repeats the last row; not stored)
        int64_t row = mb + m;
        if (a.gather) row = a.gather[row];
        xrow[i] = (const float *)a.x + row * a.ldx + 4 * (t & 15);
    }
    struct Step {
        l_u32x4 w[2], x[XL];
    };
    auto gload = [&](Step &f, int step) {
        const int k0 = KSTEP * min(first + step, steps - 1);
#pragma unroll
        for (int i = 0; i < 2; i++) f.w[i] = *(const l_u32x4 *)(wrow[i] + k0);
#pragma unroll
        for (int i = 0; i < XL; i++) f.x[i] = *(const l_u32x4 *)(xrow[i] + k0);
        __builtin_amdgcn_sched_barrier(0);  // (requests stay in the order of the steps: a step's wait leaves the next one's under way)
    };
    auto to_lds = [&](const Step &f, int buffer) {
        l_u32x4 *s_w = (l_u32x4 *)(s_raw + (2 * part + buffer) * BUFFER), *s_x = s_w + T * 8;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int r = (t >> 3) + 32 * i;
            s_w[r * 8 + ((t & 7) ^ gemm_swz(r))] = f.w[i];
        }
#pragma unroll
        for (int i = 0; i < XL; i++) {
            const int r = (t >> 4) + 16 * i;
            s_x[r * 16 + ((t & 15) ^ (r & 15))] = f.x[i];
        }
        l_lds_barrier();
    };
    // inputs 8 c .. 8 c + 7 of a step, of row r of W and of X
    auto weights = [&](int buffer, int r, int c) {
        return __builtin_bit_cast(l_bf16x8, ((const l_u32x4 *)(s_raw + (2 * part + buffer) * BUFFER))[r * 8 + (c ^ gemm_swz(r))]);
    };
    auto parts = [&](int buffer, int r, int c) {
        const l_u32x4 *s_x = (const l_u32x4 *)(s_raw + (2 * part + buffer) * BUFFER) + T * 8;
        return gemm_split(__builtin_bit_cast(float4, s_x[r * 16 + ((2 * c) ^ (r & 15))]), __builtin_bit_cast(float4, s_x[r * 16 + ((2 * c + 1) ^ (r & 15))]));
    };
    l_f32x16 mine[1][1];
    float *own;
    Step f;
    gload(f, 0);
    if constexpr (SHORT) {
        l_f32x16 quarter[4];  // (of a step's inputs, as the wavefronts have them otherwise: the same sums)
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int r = 0; r < 16; r++) quarter[kk][r] = 0.0f;
        for (int u = 0; u < steps; u++) {
            to_lds(f, u & 1);
            if (u + 1 < steps) gload(f, u + 1);
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                const int c = 2 * kk + (lane >> 5);
                const l_bf16x8 A = weights(u & 1, 32 * (wave / JM) + (lane & 31), c);
                const GemmParts B = parts(u & 1, 32 * (wave % JM) + (lane & 31), c);
#pragma unroll
                for (int p = 2; p >= 0; p--) quarter[kk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A, B.part[p], quarter[kk], 0, 0, 0);
            }
        }
        mine[0][0] = quarter[0] + quarter[1] + quarter[2] + quarter[3];
        l_lds_barrier();
        own = (float *)s_raw + gemm_epilogue_floats(1, 1) * wave;
    } else {
        l_f32x16 acc[2][JM], total[2][JM];
        auto clear = [&](l_f32x16(&v)[2][JM]) {
#pragma unroll
            for (int o = 0; o < 2 * JM; o++)
#pragma unroll
                for (int r = 0; r < 16; r++) v[o / JM][o % JM][r] = 0.0f;
        };
        auto run = [&](Step &f, int step, int buffer) {
            to_lds(f, buffer);
            gload(f, step + 1);
            if (KS > 1 && first + step >= steps) return;
            // (a wavefront takes a quarter of the step's inputs)
            const int c = 2 * wave + (lane >> 5);
            l_bf16x8 A[2];
            GemmParts B[JM];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                A[i] = weights(buffer, 32 * i + (lane & 31), c);
                if (i < JM) B[i] = parts(buffer, 32 * i + (lane & 31), c);
            }
#pragma unroll
            for (int p = 2; p >= 0; p--)  // (the small parts first)
#pragma unroll
                for (int o = 0; o < 2 * JM; o++)
                    acc[o / JM][o % JM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[o / JM], B[o % JM].part[p], acc[o / JM][o % JM], 0, 0, 0);
        };
        clear(total);
        clear(acc);
        auto fold = [&] {
#pragma unroll
            for (int o = 0; o < 2 * JM; o++) total[o / JM][o % JM] += acc[o / JM][o % JM];
            clear(acc);
        };
        const int pairs = share & ~1;
        for (int u0 = 0; u0 < pairs; u0 += FOLD) {
            const int u1 = min(u0 + FOLD, pairs);
            for (int u = u0; u < u1; u += 2) {
                run(f, u, 0);
                run(f, u + 1, 1);
            }
            fold();
        }
        if (share & 1) {
            run(f, pairs, 0);
            fold();
        }
        // the four wavefronts' sums of a 32 x 32 tile each
        l_lds_barrier();
        float4 *sums = (float4 *)s_raw;
#pragma unroll
        for (int o = 0; o < 2 * JM; o++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const l_f32x16 &v = total[o / JM][o % JM];
                sums[((o * 4 * KS + 4 * part + wave) * 4 + q) * 64 + lane] = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
            }
        l_lds_barrier();
        if (part || wave >= 2 * JM) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            float4 v = sums[(wave * 4 * KS * 4 + q) * 64 + lane];
#pragma unroll
            for (int w = 1; w < 4 * KS; w++) {
                const float4 z = sums[((wave * 4 * KS + w) * 4 + q) * 64 + lane];
                v = make_float4(v.x + z.x, v.y + z.y, v.z + z.z, v.w + z.w);
            }
            mine[0][0][4 * q] = v.x, mine[0][0][4 * q + 1] = v.y, mine[0][0][4 * q + 2] = v.z, mine[0][0][4 * q + 3] = v.w;
        }
        // (a wavefront's own quarter of s_raw: no other one reads it any more)
        static_assert(4 * gemm_epilogue_floats(1, 1) <= 16384 * KS, "the epilogue's floats lie among a wavefront's own sums");
        own = (float *)s_raw + 4096 * KS * wave;
    }
    m0 += 32 * (wave % JM), n0 += 32 * (wave / JM);
    // An infinite activation's parts are itself and NaNs, and an infinite weight times a part that is zero is one: results that are NaN are computed again, on
    // the fp32 instructions (lane l has element l / 32 of two of row l % 32; a half's eight elements of 16 are consecutive).  509 positions through two experts of
    // 4096 x 1024 of which one has an infinite weight, half of the second products: 0.61 ms as on those instructions before, 0.26 without it, 0.48 like this (8.8 as a sum a lane).
    bool nan = false;
#pragma unroll
    for (int r = 0; r < 16; r++) nan |= mine[0][0][r] != mine[0][0][r];
    if (__any(nan)) {
        const int at = lane & 31, h = 8 * (lane >> 5), m = min(m0 + at, mcount - 1);
        const uint16_t *w = W + min(n0 + at, a.n_rows - 1) * a.ld + h;
        const float *x = (const float *)a.x + (a.gather ? (int64_t)a.gather[mb + m] : mb + m) * a.ldx + h;
        l_f32x16 plain;
#pragma unroll
        for (int r = 0; r < 16; r++) plain[r] = 0.0f;
        for (int k = 0; k < a.ld; k += 16) {
            const l_u32x4 wv = *(const l_u32x4 *)(w + k);
            const float4 x0 = *(const float4 *)(x + k), x1 = *(const float4 *)(x + k + 4);
            const float xf[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int e = 0; e < 8; e++) plain = __builtin_amdgcn_mfma_f32_32x32x2f32(e & 1 ? l_bf16_hi(wv[e >> 1]) : l_bf16_lo(wv[e >> 1]), xf[e], plain, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; r++) mine[0][0][r] = mine[0][0][r] != mine[0][0][r] ? plain[r] : mine[0][0][r];
    }
    gemm_epilogue<1, EPI, 1, 1>(a, mine, own, mb, m0, mcount, n0, lane);
}

template <int EPI, bool GROUPED, int KS, int TM, bool SHORT = false>
static hipError_t gemm_parts_go(hipStream_t s, const GemmArgs &a, unsigned n_nt) {
    constexpr unsigned lds = SHORT ? 2 * (128 + 4 * TM) * 64 : KS * TM * 1024u;  // (the sums; the operands take three quarters of it, or all)
    static_assert(2 * (128 + 4 * TM) * 64 <= TM * 1024 && 4 * 4 * gemm_epilogue_floats(1, 1) <= 2 * (128 + 4 * TM) * 64, "two steps' operands lie in it; SHORT: the epilogue's floats");
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute((const void *)gemm_parts_kernel<EPI, GROUPED, KS, TM, SHORT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const dim3 grid = GROUPED ? dim3(8 * (((unsigned)a.max_tiles * n_nt + 7) / 8), L_GEMM_TILE / TM) : dim3((unsigned)((a.M + TM - 1) / TM), n_nt);
    hipLaunchKernelGGL((gemm_parts_kernel<EPI, GROUPED, KS, TM, SHORT>), grid, dim3(256 * KS), lds, s, a, n_nt);
    return hipGetLastError();
}
template <int EPI, bool GROUPED>
static hipError_t gemm_parts_launch(hipStream_t s, const GemmArgs &a, int64_t cols) {
    const unsigned n_nt = (unsigned)((cols + 63) / 64);
    // Where tiles of 64 x 64 leave a CU one workgroup: two groups of wavefronts, and where they leave half the CUs none, 32 positions a tile.  us with one
    // group, two, two and 32 positions: 509 positions, 1024 x 1024 (128 tiles) 15.2, 12.2, 9.3; x 4096: 48, 34.5, 25; x 256: 6.7, 6.8, 5.3; 2048 x 1024 (256):
    // 15.9, 12.9, 12.2; x 256: 7.3, 7.3, 6.7; 100 positions, 8192 x 1024 (256) 15.8, 12.9, 14.0; 509, 3392 x 1024 (424) 20, 23, 21.  (A matrix's last block of
    // a grouped product is half full on average.)
    const int64_t halves = GROUPED ? (a.M + 63) / 64 + a.M / (2 * max(a.rows_each, 1)) : (a.M + 63) / 64, tiles = halves * n_nt;
    // (of one or two steps, all results: see SHORT)
    if (a.ld <= 128) return gemm_parts_go<EPI, GROUPED, 1, 64, true>(s, a, n_nt);
    if constexpr (!GROUPED)
        if (tiles <= 128 || (a.ld < 512 && tiles <= 256)) return gemm_parts_go<EPI, false, 2, 32>(s, a, n_nt);
    return a.ld >= 512 && tiles <= 256 ? gemm_parts_go<EPI, GROUPED, 2, 64>(s, a, n_nt) : gemm_parts_go<EPI, GROUPED, 1, 64>(s, a, n_nt);
}

template <int PREC, int EPI>
static hipError_t gemm_launch(hipStream_t s, const GemmArgs &a) {
    // columns the epilogue covers: an activation-typed result is zeroed up to its row stride
    const bool acts = EPI == GE_ACT || EPI == GE_UP || EPI == GE_EMBED;
    const int64_t cols = EPI == GE_GLU ? 2 * a.acols : acts ? a.acols : a.n_rows;
    if (k_few_pays(a, PREC, cols)) return k_few(s, a, PREC, EPI, cols);
    if (a.tiles) {
        if (EPI != GE_STORE && EPI != GE_UP && EPI != GE_GLU) return hipErrorInvalidValue;
        constexpr int E = EPI == GE_UP || EPI == GE_GLU ? EPI : GE_STORE;
        if (PREC) return gemm_parts_launch<E, true>(s, a, cols);
        if (cols > 64)
            hipLaunchKernelGGL((gemm_kernel<E, 128, L_GEMM_TILE, true>), dim3((unsigned)a.max_tiles, (unsigned)((cols + 127) / 128)), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((gemm_kernel<E, 64, L_GEMM_TILE, true>), dim3((unsigned)a.max_tiles, (unsigned)((cols + 63) / 64)), dim3(256), 0, s, a);
        return hipGetLastError();
    }
    if (PREC) return gemm_parts_launch<EPI, false>(s, a, cols);
    // (up to two steps of 64 inputs, a tile is its loads' latency and its epilogue: four small ones a CU wait for each other less, unless there is little
    // behind the products and tiles enough.  128 inputs, us, tiles of 64 x 64 and 128 x 128: 2048 positions x 2048 rows, softplus 10.1 and 14.4, an activation 8.5 and 16.3, stored
    // 7.7 and 8.4; x 8192 rows 26 and 29, 20 and 32, 19.7 and 20.2; x 16 384 57 and 55, 37 and 54, 43 and 40; 300 x 32 000, stored 16.7 and 14.4)
    constexpr int64_t enough = EPI == GE_STORE || EPI == GE_RESID ? 640 : EPI == GE_DECAY || EPI == GE_SIGMOID ? 2048 : (int64_t)1 << 62;
    const int64_t big = ((cols + 127) / 128) * ((a.M + 127) / 128);
    if (big >= (a.ld > 128 ? 256 : enough))
        hipLaunchKernelGGL((gemm_kernel<EPI, 128, 128, false>), dim3((unsigned)((a.M + 127) / 128), (unsigned)((cols + 127) / 128)), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((gemm_kernel<EPI, 64, 64, false>), dim3((unsigned)((a.M + 63) / 64), (unsigned)((cols + 63) / 64)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t k_gemm(hipStream_t s, const GemmArgs &args, int prec, int epi) {
    GemmArgs a = args;
    if (!a.acols) a.acols = a.lda;
    if (!a.w || !a.x || a.n_rows < 1 || a.M < 1 || a.ld % 64 != 0 || a.ldx < a.ld || a.lda % 64 != 0 || a.acols % 64 != 0 ||
        a.acols > a.lda || (a.tiles && a.matrices < 1))
        return hipErrorInvalidValue;
    const bool acts = epi == GE_ACT || epi == GE_UP || epi == GE_EMBED;
    if (epi == GE_GLU ? (!a.outa || a.n_rows % 2 != 0 || 2 * a.acols < a.n_rows)
        : acts        ? (!a.outa || a.acols < a.n_rows)
                      : (!a.outf || a.ldo < a.n_rows))
        return hipErrorInvalidValue;
#define GO(E) \
    case E: return prec ? gemm_launch<1, E>(s, a) : gemm_launch<0, E>(s, a)
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

// ---------------------------------------------------------------------------------------------------------------
// rows: pending update, norm, conversion to activations
// ---------------------------------------------------------------------------------------------------------------
// NQ: quads of elements a thread holds (K a multiple of 4, at most 1024 NQ); 0: any K, element by element
template <int PREC, int NQ>
__global__ __launch_bounds__(256) void norm_rows_kernel(float *X, int K, const float *w, float eps, const float *Y, const float *yw,
                                                        float mult, const int32_t *gather, void *outa, int64_t lda) {
    __shared__ float s_red[4];
    const int64_t m = blockIdx.x, src = gather ? gather[m] : m;
    float *x = X + src * K;
    const float *y = Y ? Y + src * K : nullptr;
    const int t = threadIdx.x;
    if constexpr (NQ > 0) {
        float4 v[NQ];
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int i = 4 * (t + 256 * u);
            v[u] = i < K ? *(const float4 *)(x + i) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if (y) {
            float4 z[NQ];
            float ss = 0.0f;
#pragma unroll
            for (int u = 0; u < NQ; u++) {
                const int i = 4 * (t + 256 * u);
                z[u] = i < K ? *(const float4 *)(y + i) : make_float4(0.f, 0.f, 0.f, 0.f);
                ss = fmaf(z[u].x, z[u].x, fmaf(z[u].y, z[u].y, fmaf(z[u].z, z[u].z, fmaf(z[u].w, z[u].w, ss))));
            }
            const float f = mult / sqrtf(l_block_sum(ss, s_red) / (float)K + eps);
#pragma unroll
            for (int u = 0; u < NQ; u++) {
                const int i = 4 * (t + 256 * u);
                if (i >= K) continue;
                const float4 g = *(const float4 *)(yw + i);
                v[u].x = fmaf(f * z[u].x, g.x, v[u].x);
                v[u].y = fmaf(f * z[u].y, g.y, v[u].y);
                v[u].z = fmaf(f * z[u].z, g.z, v[u].z);
                v[u].w = fmaf(f * z[u].w, g.w, v[u].w);
                *(float4 *)(x + i) = v[u];
            }
        }
        float r = 1.0f;
        if (w) {
            float ss = 0.0f;
#pragma unroll
            for (int u = 0; u < NQ; u++) ss = fmaf(v[u].x, v[u].x, fmaf(v[u].y, v[u].y, fmaf(v[u].z, v[u].z, fmaf(v[u].w, v[u].w, ss))));
            r = 1.0f / sqrtf(l_block_sum(ss, s_red) / (float)K + eps);
        }
        if (!outa) return;
#pragma unroll
        for (int u = 0; u < NQ; u++) {
            const int i = 4 * (t + 256 * u);
            if (i >= lda) continue;
            const float4 g = w && i < K ? *(const float4 *)(w + i) : make_float4(1.f, 1.f, 1.f, 1.f);
            const float4 q = make_float4(v[u].x * r * g.x, v[u].y * r * g.y, v[u].z * r * g.z, v[u].w * r * g.w);
            if (PREC)
                *(float4 *)((float *)outa + m * lda + i) = q;
            else
                *(uint2 *)((uint16_t *)outa + m * lda + i) = make_uint2(l_pack_bf16(q.x, q.y), l_pack_bf16(q.z, q.w));
        }
        return;
    }
    float ry = 0.0f;
    if (y) {
        float ss = 0.0f;
        for (int i = t; i < K; i += 256) ss = fmaf(y[i], y[i], ss);
        ry = 1.0f / sqrtf(l_block_sum(ss, s_red) / (float)K + eps);
    }
    float r = 1.0f;
    if (w || y) {
        float ss = 0.0f;
        for (int i = t; i < K; i += 256) {
            float v = x[i];
            if (y) {
                v += mult * (y[i] * ry * yw[i]);
                x[i] = v;
            }
            ss = fmaf(v, v, ss);
        }
        if (w) r = 1.0f / sqrtf(l_block_sum(ss, s_red) / (float)K + eps);
    }
    if (!outa) return;
    for (int64_t i = t; i < lda; i += 256) {
        float v = 0.0f;
        if (i < K) v = w ? x[i] * r * w[i] : x[i];
        l_store_act<PREC>(outa, m * lda + i, v);
    }
}
hipError_t k_norm_rows(hipStream_t s, float *x, int K, int M, const float *w, float eps, const float *y, const float *yw,
                       float mult, const int32_t *gather, void *outa, int64_t lda, int prec) {
    if (M < 1 || (y && gather)) return hipErrorInvalidValue;
#define GO(N)                                                                                                                             \
    do {                                                                                                                                  \
        if (prec)                                                                                                                         \
            hipLaunchKernelGGL((norm_rows_kernel<1, N>), dim3((unsigned)M), dim3(256), 0, s, x, K, w, eps, y, yw, mult, gather, outa, lda); \
        else                                                                                                                              \
            hipLaunchKernelGGL((norm_rows_kernel<0, N>), dim3((unsigned)M), dim3(256), 0, s, x, K, w, eps, y, yw, mult, gather, outa, lda); \
    } while (0)
    // (lda, a multiple of 64, may exceed K by up to 63 columns: they are covered, too)
    const int64_t cols = std::max<int64_t>(K, outa ? lda : 0);
    if (K % 4 != 0 || cols > 8192)
        GO(0);
    else if (cols <= 1024)
        GO(1);
    else if (cols <= 2048)
        GO(2);
    else if (cols <= 4096)
        GO(4);
    else
        GO(8);
#undef GO
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// mixture of experts
// ---------------------------------------------------------------------------------------------------------------
// one workgroup per token
__global__ __launch_bounds__(64) void route_kernel(const float *z, int64_t ldz, const float *bias, int E, int top, int kind, int32_t *choice,
                                                   float *score) {
    extern __shared__ __align__(16) float s_mem[];
    __shared__ int s_sel[64];
    __shared__ float s_score[64];
    const int64_t m = blockIdx.x;
    l_route<false>(z + m * ldz, bias, E, top, kind, s_mem, s_sel, s_score);
    for (int k = threadIdx.x; k < top; k += 64) {
        choice[m * top + k] = s_sel[k];
        score[m * top + k] = s_score[k];
    }
}
hipError_t k_route(hipStream_t s, const float *z, int64_t ldz, const float *bias, int M, int E, int top, int kind, int32_t *choice,
                   float *score) {
    if (E < 1 || top < 1 || top > E || top > 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL(route_kernel, dim3((unsigned)M), dim3(64), E * sizeof(float), s, z, ldz, bias, E, top, kind, choice, score);
    return hipGetLastError();
}

// one workgroup: counts, offsets, slots and the list of tiles.  The order of an expert's slots is whatever the LDS counters
// give; every slot is computed on its own, so no result depends on it.  What bounds it is latency, so a thread's first GROUP_Q choices are
// requested together, a choice is counted once (its place among its expert's is what the counter was) and the offsets are a scan: 2048 tokens with four of
// 32 experts each 10 us, against 15; 57 tokens with four of 16 2.8 and 3.4, of 64 2.9 and 8.0; one of 2, whose offsets were no work, 2.7 and 2.5.
#define GROUP_Q 8
// sums over the lanes up to and including this one, without LDS: within the rows of sixteen lanes, then the rows before
template <int SHIFT>
__device__ __forceinline__ int group_add(int v) {
    return v + __builtin_amdgcn_update_dpp(0, v, 0x110 + SHIFT, 0xF, 0xF, true);  // row_shr
}
__device__ __forceinline__ int group_scan(int v, int lane) {
    v = group_add<8>(group_add<4>(group_add<2>(group_add<1>(v))));
    const int a = __builtin_amdgcn_readlane(v, 15), b = __builtin_amdgcn_readlane(v, 31), c = __builtin_amdgcn_readlane(v, 47);
    return v + (lane >= 16 ? a : 0) + (lane >= 32 ? b : 0) + (lane >= 48 ? c : 0);
}
// What the lists of blocks are made of: blocks of tile_rows (IMAGES: of tiles_plan.h's units, with a rule for each of two products)
struct GroupLists {
    GemmTile *tiles[2];
    int tile_rows;
    TilesRule rule[2];
};
template <bool IMAGES>
__global__ __launch_bounds__(1024) void group_kernel(const int32_t *choice, const float *score, int M, int E, int top, int32_t *slot_row,
                                                     float *slot_scale, int32_t *slot_of, int32_t *n_tiles, GroupLists lists) {
    constexpr int NP = IMAGES ? 2 : 1;
    extern __shared__ __align__(16) int s_int[];
    __shared__ int s_wave[1 + NP][16];
    int *cnt = s_int, *off = s_int + E;
    const int n = M * top, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int c[GROUP_Q], rank[GROUP_Q];
    float f[GROUP_Q];
#pragma unroll
    for (int u = 0; u < GROUP_Q; u++) {
        const int i = min(t + 1024 * u, n - 1);
        c[u] = choice[i];
        f[u] = score[i];
    }
    for (int e = t; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < GROUP_Q; u++)
        if (t + 1024 * u < n) rank[u] = atomicAdd(&cnt[c[u]], 1);
    for (int i = t + 1024 * GROUP_Q; i < n; i += 1024) slot_of[i] = atomicAdd(&cnt[choice[i]], 1);
    __syncthreads();
    // each product's bound, or whole tiles: four wavefronts add up one product's blocks of one kind each
    unsigned bound[NP];
    if constexpr (IMAGES) {
        __shared__ float s_time[4];
        const bool ask = lists.rule[0].n_cu | lists.rule[1].n_cu;
        if (ask) {
            const int w = __builtin_amdgcn_readfirstlane(wave);
            if (w < 4) {
                const TilesRule r = lists.rule[w & 1];
                int blocks = 0, weight = 0;
                for (int e = lane; e < E; e += 64) {
                    const TilesSplit v = tiles_split((unsigned)(cnt[e] + TILES_UNIT - 1) / TILES_UNIT, w < 2 ? r.bound : TILES_WHOLE_UNITS);
                    blocks += (int)v.blocks;
                    weight += (int)v.weight;
                }
                blocks = group_scan(blocks, lane);
                weight = group_scan(weight, lane);
                if (lane == 63) s_time[w] = r.n_cu ? tiles_rounds(r, (unsigned)blocks, (unsigned)weight) : 0.0f;
            }
            __syncthreads();
        }
#pragma unroll
        for (int p = 0; p < NP; p++) bound[p] = ask && s_time[2 + p] < s_time[p] ? TILES_WHOLE_UNITS : lists.rule[p].bound;
    }
    // rows and blocks of the experts before e (E <= 1024: a thread for each)
    const int rows = t < E ? cnt[t] : 0;
    const unsigned units = (unsigned)(rows + TILES_UNIT - 1) / TILES_UNIT;
    int nt[NP];
    if constexpr (IMAGES) {
#pragma unroll
        for (int p = 0; p < NP; p++) nt[p] = (int)tiles_blocks(units, bound[p]);
    } else {
        nt[0] = (rows + lists.tile_rows - 1) / lists.tile_rows;
    }
    int sr = group_scan(rows, lane), st[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) st[p] = group_scan(nt[p], lane);
    if (E > 64) {
        if (lane == 63) {
            s_wave[0][wave] = sr;
#pragma unroll
            for (int p = 0; p < NP; p++) s_wave[1 + p][wave] = st[p];
        }
        __syncthreads();
        for (int w = 0; w < wave; w++) {
            sr += s_wave[0][w];
#pragma unroll
            for (int p = 0; p < NP; p++) st[p] += s_wave[1 + p][w];
        }
    }
    if (t < E) {
        off[t] = sr - rows;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            GemmTile *tiles = lists.tiles[p] + (st[p] - nt[p]);
            const TilesShares share(IMAGES ? units : 0, IMAGES ? (unsigned)nt[p] : 0);
            for (int k = 0, r0 = 0; k < nt[p]; k++) {
                const int r1 = IMAGES ? TILES_UNIT * (int)share.at((unsigned)k + 1) : r0 + lists.tile_rows;
                tiles[k] = GemmTile{t, sr - rows + r0, min(r1, rows) - r0};
                r0 = r1;
            }
            if (t == E - 1) n_tiles[p] = st[p];
        }
    }
    __syncthreads();
    auto put = [&](int i, int expert, float scale, int place) {
        const int slot = off[expert] + place;
        slot_row[slot] = i / top;
        slot_scale[slot] = scale;
        slot_of[i] = slot;
    };
#pragma unroll
    for (int u = 0; u < GROUP_Q; u++)
        if (t + 1024 * u < n) put(t + 1024 * u, c[u], f[u], rank[u]);
    for (int i = t + 1024 * GROUP_Q; i < n; i += 1024) put(i, choice[i], score[i], slot_of[i]);
}
hipError_t k_group(hipStream_t s, const int32_t *choice, const float *score, int M, int E, int top, int32_t *slot_row,
                   float *slot_scale, int32_t *slot_of, GemmTile *tiles, int32_t *n_tiles, int tile_rows) {
    if (E < 1 || E > 1024 || M < 1 || top < 1 || tile_rows < 1) return hipErrorInvalidValue;
    GroupLists l = {};
    l.tiles[0] = tiles;
    l.tile_rows = tile_rows;
    hipLaunchKernelGGL(group_kernel<false>, dim3(1), dim3(1024), 2 * E * sizeof(int), s, choice, score, M, E, top, slot_row, slot_scale, slot_of, n_tiles, l);
    return hipGetLastError();
}
hipError_t k_group_images(hipStream_t s, const int32_t *choice, const float *score, int M, int E, int top, int32_t *slot_row, float *slot_scale,
                          int32_t *slot_of, GemmTile *const tiles[2], int32_t *n_tiles, const TilesRule rule[2]) {
    if (E < 1 || E > 1024 || M < 1 || top < 1 || rule[0].bound < 1 || rule[0].bound > TILES_MAX_UNITS || rule[1].bound < 1 || rule[1].bound > TILES_MAX_UNITS) return hipErrorInvalidValue;
    const GroupLists l = {{tiles[0], tiles[1]}, 0, {rule[0], rule[1]}};
    hipLaunchKernelGGL(group_kernel<true>, dim3(1), dim3(1024), 2 * E * sizeof(int), s, choice, score, M, E, top, slot_row, slot_scale, slot_of, n_tiles, l);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void gather_add_kernel(float *x, const float *y, const int32_t *slot_of, int top, int K, float mult) {
    const int64_t m = blockIdx.y;
    const int i = 4 * (blockIdx.x * 256 + threadIdx.x);
    if (i >= K) return;
    if (K % 4 == 0) {
        const float4 a = *(const float4 *)(x + m * K + i);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
        for (int k = 0; k < top; k++) {
            const float4 q = *(const float4 *)(y + (int64_t)slot_of[m * top + k] * K + i);
            v.x += q.x;
            v.y += q.y;
            v.z += q.z;
            v.w += q.w;
        }
        *(float4 *)(x + m * K + i) = make_float4(fmaf(mult, v.x, a.x), fmaf(mult, v.y, a.y), fmaf(mult, v.z, a.z), fmaf(mult, v.w, a.w));
        return;
    }
    for (int e = i; e < min(i + 4, K); e++) {
        float v = 0.0f;
        for (int k = 0; k < top; k++) v += y[(int64_t)slot_of[m * top + k] * K + e];
        x[m * K + e] = fmaf(mult, v, x[m * K + e]);
    }
}
hipError_t k_gather_add(hipStream_t s, float *x, const float *y, const int32_t *slot_of, int M, int top, int K, float mult) {
    hipLaunchKernelGGL(gather_add_kernel, dim3((unsigned)((K + 1023) / 1024), (unsigned)M), dim3(256), 0, s, x, y, slot_of, top, K, mult);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void stream_add_kernel(float *x, const float *a, const float *b, int K) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= K) return;
    const int64_t at = (int64_t)blockIdx.y * K + i;
    x[at] = (a ? x[at] + a[at] : x[at]) + b[i];
}
hipError_t k_stream_add(hipStream_t s, float *x, const float *a, const float *b, int M, int K) {
    hipLaunchKernelGGL(stream_add_kernel, dim3((unsigned)((K + 255) / 256), (unsigned)M), dim3(256), 0, s, x, a, b, K);
    return hipGetLastError();
}

template <int PREC>
__global__ __launch_bounds__(256) void embed_rows_kernel(const float *v, int N, int act, const uint16_t *emb, int64_t emb_ld,
                                                         const int32_t *tokens, void *outa, int64_t lda) {
    const int64_t m = blockIdx.y;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= lda) return;
    l_store_act<PREC>(outa, m * lda + i, i < N ? l_act(act, v[m * N + i]) * l_bf16(emb[(int64_t)tokens[m] * emb_ld + i]) : 0.0f);
}
hipError_t k_embed_rows(hipStream_t s, const float *v, int M, int N, int act, const uint16_t *emb, int64_t emb_ld,
                        const int32_t *tokens, void *outa, int64_t lda, int prec) {
    const dim3 grid((unsigned)((lda + 255) / 256), (unsigned)M);
    if (prec)
        hipLaunchKernelGGL((embed_rows_kernel<1>), grid, dim3(256), 0, s, v, N, act, emb, emb_ld, tokens, outa, lda);
    else
        hipLaunchKernelGGL((embed_rows_kernel<0>), grid, dim3(256), 0, s, v, N, act, emb, emb_ld, tokens, outa, lda);
    return hipGetLastError();
}
