// Device helpers of the layered models' kernels.
#pragma once

#include "dev_common.h"
#include "layered.h"

typedef __bf16 l_bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t l_pack_bf16(float a, float b) {
    l_bf16x2 v;
    v.x = (__bf16)a;
    v.y = (__bf16)b;
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float l_bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float l_bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ float l_bf16(uint16_t w) { return __uint_as_float((uint32_t)w << 16); }

__device__ __forceinline__ float l_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float l_silu(float z) { return z / (1.0f + expf(-z)); }
// log(1 + exp(z)) = max(z, 0) + log(1 + e), e = exp(-|z|); log(1 + e) = 2 artanh(s), s = e / (2 + e) <= 1/3, by its power series
// (the first term left out is 2 s^17 / 17 < 1e-9 of the sum): small relative error also where the result is small
__device__ __forceinline__ float l_softplus(float z) {
    const float e = expf(-fabsf(z)), s = e / (2.0f + e), q = s * s;
    float p = fmaf(q, 1.0f / 15.0f, 1.0f / 13.0f);
    p = fmaf(p, q, 1.0f / 11.0f);
    p = fmaf(p, q, 1.0f / 9.0f);
    p = fmaf(p, q, 1.0f / 7.0f);
    p = fmaf(p, q, 1.0f / 5.0f);
    p = fmaf(p, q, 1.0f / 3.0f);
    p = fmaf(p, q, 1.0f);
    return fmaf(2.0f * s, p, fmaxf(z, 0.0f));
}
__device__ __forceinline__ float l_act(int act, float z) {
    if (act == LACT_RELU2) {
        const float r = fmaxf(z, 0.0f);
        return r * r;
    }
    if (act == LACT_RELU) return fmaxf(z, 0.0f);
    if (act == LACT_SILU) return l_silu(z);
    if (act == LACT_GELU_TANH) return 0.5f * z * (1.0f + tanhf(0.797884560802865356f * fmaf(0.044715f * z * z, z, z)));
    return 0.5f * z * (1.0f + erff(z * 0.707106781186547524f));
}
// erf by formula 7.1.26 of Abramowitz and Stegun, Handbook of Mathematical Functions: within 1.5e-7 everywhere, a dozen
// instructions; for results that are rounded to bf16
__device__ __forceinline__ float l_erf_short(float x) {
    const float a = fabsf(x), t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, a, 1.0f));
    float p = fmaf(1.061405429f, t, -1.453152027f);
    p = fmaf(p, t, 1.421413741f);
    p = fmaf(p, t, -0.284496736f);
    p = fmaf(p, t, 0.254829592f);
    return copysignf(1.0f - p * t * __builtin_amdgcn_exp2f(-1.44269504088896341f * a * a), x);
}
// the activation of a result of the given precision
template <int PREC>
__device__ __forceinline__ float l_act_rounded(int act, float z) {
    if (PREC == 0 && act == LACT_GELU_ERF) return 0.5f * z * (1.0f + l_erf_short(z * 0.707106781186547524f));
    return l_act(act, z);
}

// 1 / sqrt(x) within a unit in the last place: the hardware's with a step of Newton's method.  (1 / sqrtf(x), with its exact root and quotient, is forty
// instructions in a row, which a launch of a decode step also has to fetch: 0.1 us of 3.)  The hardware takes numbers below 2^-126 for zero: small ones go in
// 2^32 times as large, which is exact.
__device__ __forceinline__ float l_rsqrt(float x) {
    const bool small = x < 0x1p-100f;
    const float v = small ? x * 0x1p32f : x;
    const float y = __builtin_amdgcn_rsqf(v), e = fmaf(-v * y, y, 1.0f), z = fmaf(0.5f * y, e, y), r = e == e ? z : y;  // (0 and infinity as they are)
    return small ? r * 0x1p16f : r;
}

// v plus its value in another lane of the same sixteen
template <int CTRL>
__device__ __forceinline__ float l_dpp_add(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// Sum over the wavefront, in every lane: sixteen lanes by DPP, the four sums of those on the scalar path (no LDS: six exchanges through it take 0.2 us,
// and a launch of a decode step has two to four such sums one after the other).
__device__ __forceinline__ float l_wave_sum(float v) {
    v = l_dpp_add<0x121>(l_dpp_add<0x122>(l_dpp_add<0x124>(l_dpp_add<0x128>(v))));  // row_ror: 8, 4, 2, 1
    const int i = __float_as_int(v);
    const float a = __int_as_float(__builtin_amdgcn_readlane(i, 0)), b = __int_as_float(__builtin_amdgcn_readlane(i, 16)),
                c = __int_as_float(__builtin_amdgcn_readlane(i, 32)), d = __int_as_float(__builtin_amdgcn_readlane(i, 48));
    return (a + b) + (c + d);
}
// sum over the workgroup; `red` holds one float per wavefront; every thread gets the total
__device__ __forceinline__ float l_block_sum(float v, float *red) {
    const int nw = (blockDim.x + 63) >> 6;
    v = l_wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.0f;
    for (int w = 0; w < nw; w++) t += red[w];
    return t;
}

// a barrier that orders LDS traffic only: what the wavefronts have under way to and from memory stays under way
__device__ __forceinline__ void l_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// l_block_sum with such a barrier; `red` is not used again behind it
__device__ __forceinline__ float l_block_sum_lds(float v, float *red) {
    const int nw = (blockDim.x + 63) >> 6;
    v = l_wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    l_lds_barrier();
    float t = 0.0f;
    for (int w = 0; w < nw; w++) t += red[w];
    return t;
}

// activations: bf16 or fp32 elements behind one pointer
template <int PREC>
__device__ __forceinline__ void l_store_act(void *p, int64_t i, float v) {
    if (PREC)
        ((float *)p)[i] = v;
    else
        ((__bf16 *)p)[i] = (__bf16)v;
}

// Rotation of the pairs (2 i, 2 i + 1), or with `half` (i, i + rot / 2), i < rot / 2, of one head at `pos` and division by the
// head's root mean square, by one wavefront.  src and dst hold D elements.
__device__ __forceinline__ void l_rotate_norm(const float *src, float *dst, int D, int rot, int half, const float *freq, int pos,
                                              int norm, float eps, int lane) {
    float ss = 0.0f;
    for (int p = lane; 2 * p < D; p += 64) {
        const bool turned = 2 * p < rot, apart = half && turned;
        const int ia = apart ? p : 2 * p, ib = apart ? p + rot / 2 : 2 * p + 1;
        float a = src[ia], b = ib < D ? src[ib] : 0.0f;
        if (turned) {
            const float ang = (float)pos * freq[p];
            const float c = cosf(ang), s = sinf(ang), u = a, v = b;
            a = u * c - v * s;
            b = v * c + u * s;
        }
        ss = fmaf(a, a, ss);
        ss = fmaf(b, b, ss);
        dst[ia] = a;
        if (ib < D) dst[ib] = b;
    }
    if (!norm) return;
    const float r = l_rsqrt(l_wave_sum(ss) / (float)D + eps);
    for (int p = lane; 2 * p < D; p += 64) {
        const bool apart = half && 2 * p < rot;
        const int ia = apart ? p : 2 * p, ib = apart ? p + rot / 2 : 2 * p + 1;
        dst[ia] *= r;
        if (ib < D) dst[ib] *= r;
    }
}

// Choice of experts by one workgroup: an expert's place among all by its logit is the number of larger ones (the lower index
// first among equals); sel[place], score[place] for the first `top` places.  zs: LDS for E logits; sel and score are LDS or
// global memory of the workgroup's own (IN_LDS: LDS, and the barriers order nothing else).
template <bool IN_LDS>
__device__ __forceinline__ void l_route(const float *z, const float *bias, int E, int top, int kind, float *zs, int *sel, float *score) {
    const int t = threadIdx.x, nt = blockDim.x;
    auto route_barrier = [] {
        if (IN_LDS)
            l_lds_barrier();
        else
            __syncthreads();
    };
    for (int e = t; e < E; e += nt) zs[e] = z[e] + (bias ? bias[e] : 0.0f);
    for (int k = t; k < top; k += nt) sel[k] = 0, score[k] = 0.0f;  // (a place that no number takes, with NaN among them, stays defined)
    route_barrier();
    for (int e = t; e < E; e += nt) {
        const float v = zs[e];
        int rank = 0;
#pragma unroll 8
        for (int o = 0; o < E; o++) rank += (zs[o] > v || (zs[o] == v && o < e)) ? 1 : 0;
        if (rank < top) {
            sel[rank] = e;
            score[rank] = kind == LROUTE_SIGMOID_IN ? l_sigmoid(v) : v;
        }
    }
    route_barrier();
    if (kind == LROUTE_SOFTMAX_OUT) {
        if (t < 64) {  // (top <= 64)
            const float v = t < top ? score[t] : -INFINITY, m = wave_max_f32(v);
            const float p = t < top ? expf(v - m) : 0.0f, sum = l_wave_sum(p);
            if (t < top) score[t] = p / sum;
        }
        route_barrier();
    }
}
