// Classifier rows of several prompt positions at once (the logits that a scored text wants): final rmsnorm and classifier of
// the reference's step (src/inference.jl:309,312) for up to 8 positions per pass over the classifier's weights.
//
// One position a pass is bound by the weights (128256 x 4096 q4_K or q6_K: 74 us, the stream's rate); a second position costs
// no further byte.  So a first launch normalises and quantizes the positions, each once and in its own workgroup (a step's
// classifier does it again in each of its 256), and the second holds all of them in LDS, decodes a weight's nibbles and scales
// once and multiplies them with every position.  The terms are those of the step's classifier (q8_K inputs, integer sums of a
// chunk, fp64 from there); only the order of the fp64 sum differs.
// Split: a block of a row belongs to as many neighbouring lanes as it has chunks (8; q6_K 4), so a wavefront reads 8 (16) rows,
// 128 bytes of each at a time, a row's sum costs 3 (2) exchanges instead of 6, and the lanes of different rows read one address
// of LDS.  What bounds it from 4 positions on are the vector instructions of the products.
// Measured (us a pass; a position alone 74 / 15.4 / 14.9): 4 / 8 positions of 128256 x 4096 q6_K 94 / 135, of 32000 x 2048 q4_K
// 15.3 / 22.4, of 32000 x 512 fp32 11.9 / 17.8.  (With loads past the caches the q6_K passes took 125 / 138: a line's two pieces
// were fetched twice.)
#include "matvec_dev.h"

constexpr int SCORE_THREADS = 512, SCORE_WAVES = SCORE_THREADS / 64;

template <bool KQ>
__global__ __launch_bounds__(1024) void score_stage_kernel(const float *x, ScoreRows rows, const float *normw, int K, char *images, int image) {
    __shared__ double red[16];
    PhaseArgs a{};
    a.xf = x + (int64_t)rows.row[blockIdx.x] * K;
    a.normw = normw;
    char *to = images + (int64_t)blockIdx.x * image;
    stage_activations<PRO_RMSNORM, KQ, false>(a, 0, K, (int8_t *)to, (int16_t *)(to + K), (float *)(to + K + K / 8), (float *)to, red);
}

// sums over aligned groups of LANES lanes (2, 4, 8 or 16), on every lane of the group
template <int LANES>
__device__ __forceinline__ double group_sum_f64(double v) {
    v += dpp_f64<DPP_QUAD_SWAP1>(v);
    v += dpp_f64<DPP_QUAD_SWAP2>(v);
    if (LANES >= 8) v += dpp_f64<DPP_ROW_HALF_MIRROR>(v);
    if (LANES >= 16) v += dpp_f64<DPP_ROW_MIRROR>(v);
    return v;
}

// lane `sub` of a row's LANES lanes stores positions sub, sub + LANES, ...
template <int R, int LANES>
__device__ __forceinline__ void score_store(const double (&acc)[R], int sub, int64_t row, int64_t n_rows, float *y, int n) {
    double sum[R];
#pragma unroll
    for (int p = 0; p < R; p++) sum[p] = group_sum_f64<LANES>(acc[p]);
    if (row >= n_rows) return;
#pragma unroll
    for (int p0 = 0; p0 < R; p0 += LANES) {
        double v = sum[p0];
#pragma unroll
        for (int k = 1; k < LANES && p0 + k < R; k++) v = sub == k ? sum[p0 + k] : v;
        if (p0 + sub < n && p0 + sub < R) y[(p0 + sub) * n_rows + row] = (float)v;
    }
}

__device__ __forceinline__ void score_images(uint4 *smem, const char *images, int bytes) {
    const uint4 *from = (const uint4 *)images;
    for (int i = threadIdx.x; i < bytes / 16; i += SCORE_THREADS) smem[i] = from[i];
    __syncthreads();
}

// y[p * n_rows + row] for the n <= R positions whose images lie behind each other (all R are there to be read)
template <int TYPE, int R>
__global__ __launch_bounds__(SCORE_THREADS, 4) void score_kq_kernel(DevTensor w, const char *images, int image, float *y, int n) {
    constexpr int CPB = TYPE == L2H_TYPE_Q6_K ? 4 : 8, ROWS = WAVE / CPB;
    extern __shared__ uint4 smem[];
    score_images(smem, images, R * image);
    const int lane = threadIdx.x & 63, sub = lane % CPB, nb = (int)w.nb, K = 256 * nb;
    SegPtrs t;
    t.hdr = w.hdr;
    t.qs = (const uint4 *)w.qs;
    t.qh = (const uint4 *)w.qh;
    t.sc6 = w.sc6;
    t.d6 = w.d6;
    t.nb = w.nb;
    for (int64_t r0 = ((int64_t)blockIdx.x * SCORE_WAVES + (threadIdx.x >> 6)) * ROWS; r0 < w.ne1; r0 += (int64_t)gridDim.x * SCORE_WAVES * ROWS) {
        const int64_t row = r0 + lane / CPB, there = min(row, w.ne1 - 1);
        double acc[R];
#pragma unroll
        for (int p = 0; p < R; p++) acc[p] = 0.0;
        Chunk<TYPE> c, next, after;  // two blocks are on their way while one is multiplied
        load_chunk<false>(c, t, there, sub);
        load_chunk<false>(next, t, there, CPB * min(1, nb - 1) + sub);
        for (int b = 0; b < nb; b++) {
            load_chunk<false>(after, t, there, CPB * min(b + 2, nb - 1) + sub);
#pragma unroll
            for (int p = 0; p < R; p++) {
                const int8_t *at = (const int8_t *)smem + p * image;
                const XLds x{at, (const int16_t *)(at + K), (const float *)(at + K + K / 8), nullptr};
                acc[p] += chunk_term<false>(c, CPB * b + sub, x, nullptr, nullptr, 0);
            }
            c = next;
            next = after;
        }
        score_store<R, CPB>(acc, sub, row, w.ne1, y, n);
    }
}

// F32 weights: 16 lanes a row, fp64 sums of exact products
template <int R>
__global__ __launch_bounds__(SCORE_THREADS, 4) void score_f32_kernel(DevTensor w, const char *images, int image, float *y, int n) {
    extern __shared__ uint4 smem[];
    score_images(smem, images, R * image);
    const int lane = threadIdx.x & 63, sub = lane % 16, n4 = (int)w.ne0 / 4;
    for (int64_t r0 = ((int64_t)blockIdx.x * SCORE_WAVES + (threadIdx.x >> 6)) * 4; r0 < w.ne1; r0 += (int64_t)gridDim.x * SCORE_WAVES * 4) {
        const int64_t row = r0 + lane / 16;
        const float4 *wr = (const float4 *)(w.f32 + min(row, w.ne1 - 1) * w.ne0);
        double acc[R];
#pragma unroll
        for (int p = 0; p < R; p++) acc[p] = 0.0;
        for (int i = sub; i < n4; i += 16) {
            const float4 v = wr[i];
#pragma unroll
            for (int p = 0; p < R; p++) {
                const float4 x = *(const float4 *)((const char *)smem + p * image + 16 * i);
                acc[p] = fma((double)v.x, (double)x.x, acc[p]);
                acc[p] = fma((double)v.y, (double)x.y, acc[p]);
                acc[p] = fma((double)v.z, (double)x.z, acc[p]);
                acc[p] = fma((double)v.w, (double)x.w, acc[p]);
            }
        }
        score_store<R, 16>(acc, sub, row, w.ne1, y, n);
    }
}

static int64_t score_image(const DevTensor &w) {
    const int64_t K = w.ne0;
    return w.type == L2H_TYPE_F32 ? 4 * K : (K + K / 8 + K / 64 + 15) & ~(int64_t)15;
}
// Positions of one pass: as many as keep their images within 64 KiB of LDS, so that two workgroups share a compute unit.
// 0: the vector is too long (or not in 16-byte pieces) and the positions go one at a time.
int k_score_positions(const DevTensor &w) {
    if (w.type == L2H_TYPE_F32 && w.ne0 % 4 != 0) return 0;
    const int64_t image = score_image(w);
    return 8 * image <= 64 * 1024 ? 8 : 4 * image <= 64 * 1024 ? 4 : 0;
}
int64_t k_score_image_bytes(const DevTensor &w) { return 8 * score_image(w); }

template <int R>
static hipError_t launch_score(hipStream_t s, const DevTensor &w, const char *images, float *y, int n) {
    const int image = (int)score_image(w);
    const size_t lds = (size_t)R * image;
    const int rows = SCORE_WAVES * (w.type == L2H_TYPE_F32 ? 4 : w.type == L2H_TYPE_Q6_K ? 16 : 8);
    const dim3 grid((unsigned)std::min<int64_t>(512, (w.ne1 + rows - 1) / rows));
    switch (w.type) {
    case L2H_TYPE_Q4_K: hipLaunchKernelGGL((score_kq_kernel<L2H_TYPE_Q4_K, R>), grid, dim3(SCORE_THREADS), lds, s, w, images, image, y, n); break;
    case L2H_TYPE_Q5_K: hipLaunchKernelGGL((score_kq_kernel<L2H_TYPE_Q5_K, R>), grid, dim3(SCORE_THREADS), lds, s, w, images, image, y, n); break;
    case L2H_TYPE_Q6_K: hipLaunchKernelGGL((score_kq_kernel<L2H_TYPE_Q6_K, R>), grid, dim3(SCORE_THREADS), lds, s, w, images, image, y, n); break;
    case L2H_TYPE_F32: hipLaunchKernelGGL((score_f32_kernel<R>), grid, dim3(SCORE_THREADS), lds, s, w, images, image, y, n); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t k_score(hipStream_t s, const DevTensor &w, const float *x, const ScoreRows &rows, int n, const float *normw, char *images, float *y) {
    if (n < 1 || n > k_score_positions(w)) return hipErrorInvalidValue;
    if (w.ne1 == 0) return hipSuccess;
    const int K = (int)w.ne0, image = (int)score_image(w);
    // (4 positions or fewer run with 4 images, the rest with 8; images beyond n are read and not stored)
    if (w.type == L2H_TYPE_F32)
        hipLaunchKernelGGL(score_stage_kernel<false>, dim3(n), dim3(1024), 0, s, x, rows, normw, K, images, image);
    else
        hipLaunchKernelGGL(score_stage_kernel<true>, dim3(n), dim3(1024), 0, s, x, rows, normw, K, images, image);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return n > 4 ? launch_score<8>(s, w, images, y, n) : launch_score<4>(s, w, images, y, n);
}
