// The gated feed-forward product of short prompts (k_prefill.hip has the others).
#include "matvec_dev.h"
#include "pf_tile.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct PfFewArgs {
    const uint16_t *wbf;  // tiles of pf_tile.h: w1 row u, w3 row u = rows 2u, 2u + 1
    int64_t K;
    const uint16_t *act;  // bf16 [M][K]
    int M;
    uint16_t *hb;  // bf16 [M][ldb], column row / 2
    int64_t ldb;
};

// The w1/w3 product where whole row groups would leave most CUs without one, and a CU pulls no more than about 50 GB/s from HBM: a
// workgroup takes 32 T rows and 32 T positions, its eight wavefronts an eighth of the inputs each, and their sums are added in LDS,
// always in the same order.  A lane's operands go from memory straight to its registers, one step of 64 inputs ahead of the
// products: its weight row's chunks, which lie in one block of 4 KB of the tile for 32 rows, and its position's inputs, from the L2.
// (16384 rows x 2048 inputs, 37 positions, 64 x 64 results a workgroup: 22.3 us without the step ahead, 21.3 with it, 33.5 in
// 256-row tiles; positions laid out 64 inputs at a time, so that a load takes whole lines of them: no faster.)
template <int T>
__global__ __launch_bounds__(512, T == 1 ? 4 : 2) void pf_few_kernel(PfFewArgs a, unsigned n_mt, unsigned n_items, unsigned per) {
    constexpr int TILE = 8 * 33;  // 16-byte words of 32 x 32 results: row quad q of position p at 33 q + p
    __shared__ f32x4 s_sum[4][T * T * TILE];
    const unsigned item = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (item >= n_items) return;
    const int64_t n0 = (int64_t)(item / n_mt) * 32 * T;
    const int m0 = (int)(item % n_mt) * 32 * T, t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nk = (int)(a.K >> 6), u0 = nk * wave / 8, u1 = nk * (wave + 1) / 8;
    const int r0 = (int)(n0 & 255) + (lane & 31);
    const uint16_t *wt = a.wbf + (n0 >> 8) * (a.K >> 6) * 16384, *xp[T];
    unsigned at[T][4];
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
        for (int kk = 0; kk < 4; kk++) at[i][kk] = 8 * (8 * (r0 + 32 * i) + ((2 * kk + (lane >> 5)) ^ pf_swz(r0 + 32 * i)));
#pragma unroll
    for (int j = 0; j < T; j++) xp[j] = a.act + (int64_t)min(m0 + 32 * j + (lane & 31), a.M - 1) * a.K + 8 * (lane >> 5);
    f32x16 acc[T][T];
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
        for (int j = 0; j < T; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;
    bf16x8 A[T][4], B[T][4], An[T][4], Bn[T][4];
    auto fetch = [&](bf16x8(&A)[T][4], bf16x8(&B)[T][4], int u) {
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
#pragma unroll
            for (int i = 0; i < T; i++) A[i][kk] = *(const bf16x8 *)(wt + (int64_t)u * 16384 + at[i][kk]);
#pragma unroll
            for (int j = 0; j < T; j++) B[j][kk] = *(const bf16x8 *)(xp[j] + 64 * u + 16 * kk);
        }
    };
    auto multiply = [&] {
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int i = 0; i < T; i++)
#pragma unroll
                for (int j = 0; j < T; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(A[i][kk], B[j][kk], acc[i][j], 0, 0, 0);
    };
    if (u0 < u1) {
        fetch(A, B, u0);
        for (int u = u0; u + 1 < u1; u++) {
            fetch(An, Bn, u + 1);
            multiply();
#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
#pragma unroll
                for (int i = 0; i < T; i++) A[i][kk] = An[i][kk];
#pragma unroll
                for (int j = 0; j < T; j++) B[j][kk] = Bn[j][kk];
            }
        }
        multiply();
    }
    // wavefronts 4 .. 7 hand theirs to 0 .. 3, which then lay out one set each
    const int p = lane & 31, q = lane >> 5;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if ((wave < 4) == (half == 1)) {
#pragma unroll
            for (int i = 0; i < T; i++)
#pragma unroll
                for (int j = 0; j < T; j++)
#pragma unroll
                    for (int rq = 0; rq < 4; rq++) {
                        f32x4 v = {acc[i][j][4 * rq], acc[i][j][4 * rq + 1], acc[i][j][4 * rq + 2], acc[i][j][4 * rq + 3]};
                        f32x4 &dst = s_sum[wave & 3][(i * T + j) * TILE + 33 * (2 * rq + q) + p];
                        if (half) v += dst;
                        dst = v;
                    }
        }
        __syncthreads();
    }
    for (int o = t; o < T * T * 256; o += 512) {  // row quads of a position side by side
        const int rq = o % (8 * T), m = o / (8 * T), w = ((rq >> 3) * T + (m >> 5)) * TILE + 33 * (rq & 7) + (m & 31);
        const f32x4 v = (s_sum[0][w] + s_sum[1][w]) + (s_sum[2][w] + s_sum[3][w]);
        if (m0 + m < a.M)  // (w1 row u, w3 row u) = logical rows (2u, 2u+1), src/inference.jl:295-299
            *(uint32_t *)(a.hb + (int64_t)(m0 + m) * a.ldb + ((n0 + 4 * rq) >> 1)) = pack_bf16(swiglu_val(v.x, v.y), swiglu_val(v.z, v.w));
    }
}

// w1/w3 rows in turn, expanded by k_pf_expand: hb[m][u] = swiglu of rows 2u and 2u + 1.  The inputs' sum is formed in eight parts,
// unlike k_pf_gemm's, which is the same bit for bit from the quantized blocks: for passes that form other sums their own way too.
//
// Chosen where its tiles of 64 x 64 results are at most one a CU.  Microseconds in 256-row tiles and like this, rows x inputs: 16384 x
// 2048: 8, 37, 64 positions 28.9, 33.3, 35.0 and 15.7, 20.9, 23.8, but beyond one tile a CU 128 positions 38.6 and 38.5; 16384 x 3072:
// 39.5, 45.2, 47.6 and 21.1, 29.3, 34.5; 4096 x 1024: 64 and 256 positions 21.3, 23.0 and 6.9, 11.3; 28672 x 4096,
// 37 positions (448 tiles): 62.8 and 69.2.  Tiles of 32 x 32 where the positions fit one of those or where the larger ones are at most half
// the CUs: 4096 x 1024, 96 positions (128 tiles): 9.8, against 10.8; 200 (256 tiles): 14.7 and 10.5; 16384 x 2048, 16: 17.6 and 19.2.
// (rows: twice hidden_dim, which is a multiple of 64 where there is a bf16 copy.)
static int64_t pf_few_tiles(int64_t rows, int M, int side) { return (rows / side) * ((M + side - 1) / side); }
bool k_pf_few_pays(int64_t rows, int M) { return pf_few_tiles(rows, M, 64) <= 256; }
hipError_t k_pf_few(hipStream_t s, const uint16_t *wbf, int64_t rows, const uint16_t *act, int M, int64_t K, uint16_t *hb, int64_t ldb) {
    if (rows % 64 != 0 || K % 64 != 0 || M < 1 || ldb % 2 != 0) return hipErrorInvalidValue;
    const PfFewArgs a = {wbf, K, act, M, hb, ldb};
    const bool small = M <= 16 || pf_few_tiles(rows, M, 64) <= 128;
    const int side = small ? 32 : 64;
    const unsigned n_mt = (unsigned)((M + side - 1) / side), n_items = (unsigned)pf_few_tiles(rows, M, side), per = (n_items + 7) / 8;
    if (small)
        hipLaunchKernelGGL(pf_few_kernel<1>, dim3(8 * per), dim3(512), 0, s, a, n_mt, n_items, per);
    else
        hipLaunchKernelGGL(pf_few_kernel<2>, dim3(8 * per), dim3(512), 0, s, a, n_mt, n_items, per);
    return hipGetLastError();
}
