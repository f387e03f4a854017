// The products of k_gemm.hip for few positions, few rows, or both: C[m][n] = sum_k X[m][k] W[n][k] where tiles of 64 x 64 results
// would leave most of the chip without one.
//
// What bounds such a product is reading the matrix once, so as many wavefronts as possible have a share of it under way: a
// workgroup takes 16 or 32 rows and 16 to 64 positions, its eight wavefronts an eighth of the inputs each, and their sums are
// added in LDS, in order.  Operands go from memory straight to the registers that the matrix instructions take (a lane holds 8
// consecutive inputs of one row), the next step's under way during this one's; a position's inputs come from the L2.  Measured,
// tiles of 64 x 64 and this, microseconds: 57 positions, 2048 x 10240 bf16: 237, 29; 57 x 32768 x 2048: 55, 29; a router's 16
// experts, 333 positions x 4096 inputs: 93, 13; 16 gated experts of 2048 x 2048 with 14 positions each: 94, 42.  (Three steps
// under way instead of one: no faster; what is left is the addresses, 16 rows a load, which lie a multiple of 4 KB apart.)
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

template <int PREC, int EPI>
static hipError_t few_launch(hipStream_t s, const GemmArgs &a, int64_t cols) {
    if (a.tiles) {
        if constexpr (EPI == GE_STORE || EPI == GE_UP || EPI == GE_GLU) {
            const unsigned n_nt = (unsigned)((cols + 15) / 16), most = (unsigned)a.max_tiles * n_nt;
            hipLaunchKernelGGL((few_grouped_kernel<PREC, EPI>), dim3(8 * ((most + 7) / 8)), dim3(64 * FEW_WAVES), 0, s, a, n_nt);
            return hipGetLastError();
        }
        return hipErrorInvalidValue;
    }
#define GO(RN, JM)                                                                                                                        \
    do {                                                                                                                                  \
        const unsigned n_nt = (unsigned)((cols + 16 * RN - 1) / (16 * RN)), n_mt = (unsigned)((a.M + 16 * JM - 1) / (16 * JM));          \
        hipLaunchKernelGGL((few_kernel<PREC, EPI, RN, JM>), dim3(8 * ((n_nt * n_mt + 7) / 8)), dim3(64 * FEW_WAVES), 0, s, a, n_nt, n_mt); \
        return hipGetLastError();                                                                                                         \
    } while (0)
    // 32 rows and 64 positions at a time where that gives every CU a workgroup: half the reads of the positions (fp32 products of that size go to k_gemm's tiles)
    if (a.M <= 16) GO(1, 1);
    if constexpr (PREC) {
        GO(1, 2);
    } else {
        if (a.M <= 32 || ((cols + 31) / 32) * ((a.M + 63) / 64) < 256) GO(1, 2);
        GO(2, 4);
    }
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
