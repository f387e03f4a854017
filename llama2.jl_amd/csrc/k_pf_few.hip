// The gated feed-forward product of short prompts (k_prefill.hip has the others).
#include "matvec_dev.h"
#include "few_ring.h"

struct PfFewArgs {
    const uint16_t *wbf;  // tiles of pf_tile.h: w1 row u, w3 row u = rows 2u, 2u + 1
    int64_t K;
    const uint16_t *act;  // bf16 [M][K]
    int M;
    uint16_t *hb;  // bf16 [M][ldb], column row / 2
    int64_t ldb;
};

// The w1/w3 product where whole row groups would leave most CUs without one, and a CU pulls no more than about 70 GB/s: tiles of TN rows x TM positions, see
// few_ring.h.  The copy's tiles have a row block's step in one run of 4 or 8 KB.
template <int TN, int TM>
__global__ __launch_bounds__(256) void pf_few_kernel(PfFewArgs a, unsigned n_mt, unsigned n_items, unsigned per) {
    extern __shared__ __align__(16) unsigned char s_ring[];
    const unsigned item = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || item >= n_items) return;
    const int64_t n0 = (int64_t)(item / n_mt) * TN, nk = a.K >> 6;
    const int m0 = (int)(item % n_mt) * TM, t = threadIdx.x, lane = t & 63;
    const uint16_t *wp = a.wbf + (n0 >> 8) * nk * 16384 + 64 * (n0 & 255) + 8 * lane, *xp[TM / 8];
#pragma unroll
    for (int i = 0; i < TM / 8; i++) xp[i] = a.act + (int64_t)min(m0 + few_ring_row(i, lane), a.M - 1) * a.K + 8 * few_ring_chunk(i, lane);
    few_ring<TN, TM, FewEighths>((int)nk, blockIdx.x >> 3, s_ring, [&](int i, int k) { return wp + (int64_t)k * 16384 + 512 * i; }, [&](int i, int k) { return xp[i] + 64 * k; });
    for (int o = t; o < TM * TN / 4; o += 256) {  // row quads of a position side by side
        const int m = o / (TN / 4), rq = o % (TN / 4);
        const float4 v = few_ring_sum<TN, TM>(s_ring, m, rq);
        if (m0 + m < a.M)  // (w1 row u, w3 row u) = logical rows (2u, 2u+1), src/inference.jl:295-299
            *(uint32_t *)(a.hb + (int64_t)(m0 + m) * a.ldb + ((n0 + 4 * rq) >> 1)) = pack_bf16(swiglu_val(v.x, v.y), swiglu_val(v.z, v.w));
    }
}
template <int TN, int TM>
static hipError_t pf_few_go(hipStream_t s, const PfFewArgs &a, int64_t rows) {
    static bool set[FEW_RING_DEVICES] = {};
    const unsigned n_mt = (unsigned)((a.M + TM - 1) / TM), n_items = (unsigned)(rows / TN) * n_mt, per = (n_items + 7) / 8;
    return few_ring_go(s, pf_few_kernel<TN, TM>, set, few_ring_lds(TN, TM), 8 * per, a, n_mt, n_items, per);
}

// The same sums for few inputs, or few rows and positions, where the ring has little to bring and only its latency counts: tiles of 32 T rows x 32 T positions by eight
// wavefronts, an eighth of the inputs each, operands straight to registers a step of 64 ahead, results added in LDS in the ring's order.
template <int T>
__global__ __launch_bounds__(512, T == 1 ? 4 : 2) void pf_few_direct_kernel(PfFewArgs a, unsigned n_mt, unsigned n_items, unsigned per) {
    constexpr int TILE = FEW_RING_SUMS;
    __shared__ float4 s_sum[4][T * T * TILE];
    const unsigned item = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || item >= n_items) return;
    const int64_t n0 = (int64_t)(item / n_mt) * 32 * T;
    const int m0 = (int)(item % n_mt) * 32 * T, t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nk = (int)(a.K >> 6), u0 = nk * wave / 8, u1 = nk * (wave + 1) / 8, r0 = (int)(n0 & 255) + (lane & 31);
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
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int i = 0; i < T; i++) {
                A[i][kk] = *(const bf16x8 *)(wt + (int64_t)u * 16384 + at[i][kk]);
                B[i][kk] = *(const bf16x8 *)(xp[i] + 64 * u + 16 * kk);
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
            for (int kk = 0; kk < 4; kk++)
#pragma unroll
                for (int i = 0; i < T; i++) {
                    A[i][kk] = An[i][kk];
                    B[i][kk] = Bn[i][kk];
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
                        float4 v = make_float4(acc[i][j][4 * rq], acc[i][j][4 * rq + 1], acc[i][j][4 * rq + 2], acc[i][j][4 * rq + 3]);
                        float4 &to = s_sum[wave & 3][(i * T + j) * TILE + 33 * (2 * rq + q) + p];
                        if (half) v = make_float4(v.x + to.x, v.y + to.y, v.z + to.z, v.w + to.w);
                        to = v;
                    }
        }
        __syncthreads();
    }
    for (int o = t; o < T * T * 256; o += 512) {  // row quads of a position side by side
        const int rq = o % (8 * T), m = o / (8 * T), w = ((rq >> 3) * T + (m >> 5)) * TILE + 33 * (rq & 7) + (m & 31);
        const float4 v0 = s_sum[0][w], v1 = s_sum[1][w], v2 = s_sum[2][w], v3 = s_sum[3][w];
        if (m0 + m < a.M)
            *(uint32_t *)(a.hb + (int64_t)(m0 + m) * a.ldb + ((n0 + 4 * rq) >> 1)) =
                pack_bf16(swiglu_val((v0.x + v1.x) + (v2.x + v3.x), (v0.y + v1.y) + (v2.y + v3.y)), swiglu_val((v0.z + v1.z) + (v2.z + v3.z), (v0.w + v1.w) + (v2.w + v3.w)));
    }
}
template <int T>
static hipError_t pf_few_direct_go(hipStream_t s, const PfFewArgs &a, int64_t rows) {
    const unsigned n_mt = (unsigned)((a.M + 32 * T - 1) / (32 * T)), n_items = (unsigned)(rows / (32 * T)) * n_mt, per = (n_items + 7) / 8;
    hipLaunchKernelGGL((pf_few_direct_kernel<T>), dim3(8 * per), dim3(512), 0, s, a, n_mt, n_items, per);
    return hipGetLastError();
}

// w1/w3 rows in turn, expanded by k_pf_expand: hb[m][u] = swiglu of rows 2u and 2u + 1.  The inputs' sum is formed in eight parts,
// unlike k_pf_gemm's, which is the same bit for bit from the quantized blocks: for passes that form other sums their own way too.
//
// Chosen up to one tile of 64 x 64 results a CU.  us, rows x inputs, k_pf_gemm, this kernel as it was (operands straight to registers, eight wavefronts an eighth of the
// inputs each) and as it is, bit for bit the same: 16 384 x 2048, 8, 32 and 64 positions 27.4, 28.3, 30.6; 15.6, 20.2, 23.7; 14.7, 15.3, 17.5; 16 384 x 3072 38.2, 39.9, 43.2; 21.3,
// 28.7, 34.5; 19.8, 20.6, 23.7; 4096 x 1024, 64, 128 and 256: 18.0, 17.4, 16.8; 7.1, 10.2, 11.7; 6.1, 7.6, 9.6.  Beyond, 16 384 x 2048, 128 (512 tiles): 30.1, 38.4, 28.5; 4096 x 1024, 400
// (448): 16.4 and 16.5; 28 672 x 4096, 32 and 64 (448) 56.8, 60.8; 69.2 (37 positions); 47.0, 53.4: faster at some, but another order of the sums than such passes have had.
// The smallest tiles that come to at most one a CU, beyond that the largest that the positions fill: 4096 x 1024, 64 positions 6.1, 7.5, 7.4, 9.8 in tiles of 32 x 32, 32 x 64,
// 64 x 32 and 64 x 64, 128 (256 of 32 x 64) 10.0, 7.6, 7.5, 9.4, 256 17.9, 12.6, 12.7, 9.6; 16 384 x 2048, 32 17.6, 19.5, 15.3, 16.1.
// Up to 384 inputs, and up to 16 positions of 2048 rows, operands go to registers: 1024 x 64, 626 positions 4.3 and 5.3 through the ring; 2944 x 128, 37 3.0 and 3.5; 5248 x 256, 69 5.7 and 6.6; 1664 x
// 768, 2 4.0 and 4.6; 512 x 3264, 3 7.4 and 7.9; but 640 x 448, 267 3.9 and 3.8; 3712 x 448, 24 4.2 and 3.9; 896 x 1024, 64 5.7 and 5.1; 3840 x 2176, 3 8.3 and 7.8.
// (rows: twice hidden_dim, which is a multiple of 64 where there is a bf16 copy.)
bool k_pf_few_pays(int64_t rows, int M) { return (rows / 64) * ((M + 63) / 64) <= 256; }
hipError_t k_pf_few(hipStream_t s, const uint16_t *wbf, int64_t rows, const uint16_t *act, int M, int64_t K, uint16_t *hb, int64_t ldb) {
    if (rows % 64 != 0 || K % 64 != 0 || M < 1 || ldb % 2 != 0) return hipErrorInvalidValue;
    const PfFewArgs a = {wbf, K, act, M, hb, ldb};
    auto tiles = [&](int r, int p) { return rows / r * ((M + p - 1) / p); };
    if (K <= 384 || (M <= 16 && rows <= 2048)) return M <= 16 || tiles(64, 64) <= 128 ? pf_few_direct_go<1>(s, a, rows) : pf_few_direct_go<2>(s, a, rows);
    if (tiles(32, 32) <= 256) return pf_few_go<32, 32>(s, a, rows);
    if (M > 32 && tiles(32, 64) <= 256) return pf_few_go<32, 64>(s, a, rows);
    return M <= 32 ? pf_few_go<64, 32>(s, a, rows) : pf_few_go<64, 64>(s, a, rows);
}
