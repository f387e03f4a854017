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

// w1/w3 rows in turn, expanded by k_pf_expand: hb[m][u] = swiglu of rows 2u and 2u + 1.  The inputs' sum is formed in eight parts,
// unlike k_pf_gemm's, which is the same bit for bit from the quantized blocks: for passes that form other sums their own way too.
//
// Chosen up to one tile of 64 x 64 results a CU.  us, rows x inputs, k_pf_gemm, this kernel as it was (operands straight to registers, eight wavefronts an eighth of the
// inputs each) and as it is, bit for bit the same: 16 384 x 2048, 8, 32 and 64 positions 27.4, 28.3, 30.6; 15.6, 20.2, 23.7; 14.7, 15.3, 17.5; 16 384 x 3072 38.2, 39.9, 43.2; 21.3,
// 28.7, 34.5; 19.8, 20.6, 23.7; 4096 x 1024, 64, 128 and 256: 18.0, 17.4, 16.8; 7.1, 10.2, 11.7; 6.1, 7.6, 9.6.  Beyond, 16 384 x 2048, 128 (512 tiles): 30.1, 38.4, 28.5; 4096 x 1024, 400
// (448): 16.4 and 16.5; 28 672 x 4096, 32 and 64 (448) 56.8, 60.8; 69.2 (37 positions); 47.0, 53.4: faster at some, but another order of the sums than such passes have had.
// The smallest tiles that come to at most one a CU, beyond that the largest that the positions fill: 4096 x 1024, 64 positions 6.1, 7.5, 7.4, 9.8 in tiles of 32 x 32, 32 x 64,
// 64 x 32 and 64 x 64, 128 (256 of 32 x 64) 10.0, 7.6, 7.5, 9.4, 256 17.9, 12.6, 12.7, 9.6; 16 384 x 2048, 32 17.6, 19.5, 15.3, 16.1.
// (rows: twice hidden_dim, which is a multiple of 64 where there is a bf16 copy.)
bool k_pf_few_pays(int64_t rows, int M) { return (rows / 64) * ((M + 63) / 64) <= 256; }
hipError_t k_pf_few(hipStream_t s, const uint16_t *wbf, int64_t rows, const uint16_t *act, int M, int64_t K, uint16_t *hb, int64_t ldb) {
    if (rows % 64 != 0 || K % 64 != 0 || M < 1 || ldb % 2 != 0) return hipErrorInvalidValue;
    const PfFewArgs a = {wbf, K, act, M, hb, ldb};
    auto tiles = [&](int r, int p) { return rows / r * ((M + p - 1) / p); };
    if (tiles(32, 32) <= 256) return pf_few_go<32, 32>(s, a, rows);
    if (M > 32 && tiles(32, 64) <= 256) return pf_few_go<32, 64>(s, a, rows);
    return M <= 32 ? pf_few_go<64, 32>(s, a, rows) : pf_few_go<64, 64>(s, a, rows);
}
