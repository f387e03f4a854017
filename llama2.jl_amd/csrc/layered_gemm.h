// Epilogues of the many-token products of layered models.
#pragma once

#include "layered_dev.h"

// What an epilogue reads of row m and of columns L .. L + 3.  A lane reads all of it before its first store: the compiler cannot move such
// a load past a store, and a wait for it there is one for the stores before it (decays of 2048 x 2048: 29.7 us, 22.7 with the reads in front).
template <int EPI>
__device__ __forceinline__ float gemm_row(const GemmArgs &a, int64_t m) {
    return (EPI == GE_UP || EPI == GE_GLU) && a.row_scale ? a.row_scale[m] : 1.0f;
}
struct GemmCol {
    float rate[4], bias[4];
};
template <int EPI>
__device__ __forceinline__ GemmCol gemm_col(const GemmArgs &a, int64_t L) {
    GemmCol c = {};
    if (EPI != GE_DECAY) return c;
    // (matrices have fewer than 2^31 rows: 32-bit division)
    const unsigned last = (unsigned)a.n_rows - 1, h0 = min((unsigned)L, last) / (unsigned)a.hd;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const unsigned r = min((unsigned)(L + e), last);
        c.bias[e] = a.bias[r];
        c.rate[e] = a.rate[a.hd % 4 == 0 ? h0 : r / (unsigned)a.hd];
    }
    return c;
}

// results (m, L .. L + 3) of a product
template <int PREC, int EPI>
__device__ __forceinline__ void gemm_store4(const GemmArgs &a, int64_t m, int64_t L, float f, const GemmCol &col, float v0, float v1, float v2, float v3) {
    float v[4] = {v0, v1, v2, v3};
    if (EPI == GE_STORE || EPI == GE_RESID || EPI == GE_DECAY || EPI == GE_SIGMOID) {
        if (L >= a.n_rows) return;
        float *o = a.outf + m * a.ldo + L;
        auto value = [&](int e, float old) {
            if (EPI == GE_RESID) return fmaf(a.mult, v[e], old);
            if (EPI == GE_DECAY) return -col.rate[e] * l_softplus(v[e] + col.bias[e]);
            if (EPI == GE_SIGMOID) return l_sigmoid(v[e]);
            return v[e];
        };
        if (a.ldo % 4 == 0 && L + 3 < a.n_rows) {
            float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
            if (EPI == GE_RESID) q = *(const float4 *)o;
            *(float4 *)o = make_float4(value(0, q.x), value(1, q.y), value(2, q.z), value(3, q.w));
            return;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (L + e >= a.n_rows) break;
            o[e] = value(e, EPI == GE_RESID ? o[e] : 0.0f);
        }
    } else if (EPI == GE_GLU) {
        // (n_rows even: pairs are whole)
        const int64_t i = L >> 1;
        if (i >= a.acols) return;
        float o[2] = {0.0f, 0.0f};
        const float fi = a.scale_in ? f : 1.0f, fo = a.scale_in ? 1.0f : f;
#pragma unroll
        for (int e = 0; e < 2; e++)
            if (L + 2 * e < a.n_rows) o[e] = fo * l_act_rounded<PREC>(a.act, fi * v[2 * e]) * (fi * v[2 * e + 1]);
        if (PREC)
            *(float2 *)((float *)a.outa + m * a.lda + i) = make_float2(o[0], o[1]);
        else
            *(uint32_t *)((uint16_t *)a.outa + m * a.lda + i) = l_pack_bf16(o[0], o[1]);
    } else {
        if (L >= a.acols) return;  // (acols a multiple of 64: whole groups of four)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (L + e >= a.n_rows) {
                v[e] = 0.0f;
                continue;
            }
            if (EPI == GE_UP)
                v[e] = a.scale_in ? l_act_rounded<PREC>(a.act, f * v[e]) : f * l_act_rounded<PREC>(a.act, v[e]);
            else if (EPI == GE_EMBED)
                v[e] = l_act_rounded<PREC>(a.act, v[e]) * l_bf16(a.emb[(int64_t)a.tokens[m] * a.emb_ld + L + e]);
            else
                v[e] = l_act_rounded<PREC>(a.act, v[e]);
        }
        if (PREC)
            *(float4 *)((float *)a.outa + m * a.lda + L) = make_float4(v[0], v[1], v[2], v[3]);
        else
            *(uint2 *)((uint16_t *)a.outa + m * a.lda + L) = make_uint2(l_pack_bf16(v[0], v[1]), l_pack_bf16(v[2], v[3]));
    }
}

// The results of a wavefront, 32 NI columns from `n` x 32 NJ positions from `m` of a block of mcount that starts at row mb, as the products of 32 x 32
// leave them: register 4 rq + r of tile (i, j) is column 32 i + 8 rq + 4 (lane / 32) + r of position 32 j + lane % 32.
//
// They go through LDS, 32 positions at a time, so that the epilogue's code is there once, in a loop, and consecutive lanes store
// consecutive columns.  Unrolled over the registers, with every activation in each of 128 places, it was fetched from memory as it ran:
// 92 us of the 143 that 192 tiles of 256 x 256 results and 2048 inputs took (a gelu behind a router's factor).  Kernels before and after, us:
// those tiles 143 -> 73; a dense 8192 x 2048 activation of 2048 positions 119 -> 82; gated 28 672 x 4096 500 -> 463; plain stores of
// experts' down products 86 -> 72 and 230 -> 212; decays 22.7 -> 16.2.
// s: gemm_epilogue_floats(NI, NJ) floats of this wavefront's own.
typedef float gemm_f32x16 __attribute__((ext_vector_type(16)));
constexpr int gemm_epilogue_floats(int ni, int nj) { return 32 * (32 * ni + 4) + 32 * nj; }
template <int PREC, int EPI, int NI, int NJ>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs &a, gemm_f32x16 (&acc)[NI][NJ], float *s, int64_t mb, int m, int mcount, int64_t n, int lane) {
    constexpr int LD = 32 * NI + 4, QL = 8 * NI, STEP = 64 / QL;  // (4 modulo 64 banks, or 36: 16 lanes' quads fall into different banks)
    float *s_f = s + 32 * LD;
    const int64_t L = n + 4 * (lane & (QL - 1));
    const GemmCol col = gemm_col<EPI>(a, L);
#pragma unroll
    for (int i = 0; i < (32 * NJ + 63) / 64; i++)
        if (64 * i + lane < 32 * NJ) s_f[64 * i + lane] = gemm_row<EPI>(a, mb + min(m + 64 * i + lane, mcount - 1));
#pragma nounroll
    for (int j = 0; j < NJ; j++) {
        if (m + 32 * j >= mcount) break;
#pragma unroll
        for (int jj = 0; jj < NJ; jj++)
            if (jj == j) {
#pragma unroll
                for (int i = 0; i < NI; i++)
#pragma unroll
                    for (int rq = 0; rq < 4; rq++)
                        *(float4 *)(s + (lane & 31) * LD + 32 * i + 8 * rq + 4 * (lane >> 5)) =
                            make_float4(acc[i][jj][4 * rq], acc[i][jj][4 * rq + 1], acc[i][jj][4 * rq + 2], acc[i][jj][4 * rq + 3]);
            }
        // (one wavefront's LDS accesses are served in order; the compiler is to leave them in theirs)
        asm volatile("" ::: "memory");
#pragma nounroll
        for (int p = lane / QL; p < 32; p += STEP) {
            const float f = s_f[32 * j + p];
            asm volatile("" ::: "memory");  // (the quad's read is the last one under way: a wait for it is a wait for everything)
            const float4 v = *(const float4 *)(s + p * LD + 4 * (lane & (QL - 1)));
            if (m + 32 * j + p < mcount) gemm_store4<PREC, EPI>(a, mb + m + 32 * j + p, L, f, col, v.x, v.y, v.z, v.w);
        }
        asm volatile("" ::: "memory");
    }
}
