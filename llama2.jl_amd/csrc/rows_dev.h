// One token through a bf16 matrix, the body of a workgroup (k_rows.hip has the kernels of one product, k_step.hip those of a product
// beside something else).
#pragma once

#include "layered_dev.h"
#include "rows_plan.h"

#define ROWS_MAX_EXPERTS 1024
#define ROWS_MAX_TOP 64
#define ROWS_CHOOSE 40

// element e of the staged vector: the two halves of every group of 8 lie in separate planes, so that the lanes of a
// wavefront, each reading 8 consecutive elements as two 16-byte words, touch consecutive words
__device__ __forceinline__ int xs_index(int e, int plane) { return ((e >> 2) & 1) * plane + ((e >> 3) << 2) + (e & 3); }

// one 16-byte chunk of each of a pair of rows against the staged vector
struct RowsChunk {
    uint4 p, q;
};
typedef uint32_t rows_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 rows_word(const uint16_t *w) {
    const rows_u32x4 v = __builtin_nontemporal_load((const rows_u32x4 *)w);
    return make_uint4(v.x, v.y, v.z, v.w);
}
// (no load is skipped: how many are under way has to be known when the code is compiled for a wait to leave the later ones alone)
__device__ __forceinline__ void rows_load(RowsChunk &c, const uint16_t *w0, const uint16_t *w1, int k, int ld) {
    const unsigned at = 2u * (unsigned)min(k, ld - 8);  // (bytes: one 32-bit offset a lane behind two addresses of the wavefront's)
    c.p = rows_word((const uint16_t *)((const char *)w0 + at));
    c.q = rows_word((const uint16_t *)((const char *)w1 + at));
}
// (lanes beyond the row drop what they have added: no branch, whose other side would have to be fetched, too)
__device__ __forceinline__ void rows_fma(const RowsChunk &c, const float *xv, int plane, int k, int ld, float &acc0, float &acc1) {
    const uint4 p = c.p, q = c.q;
    const int at = min(k, ld - 8) >> 1;
    const float4 xa = *(const float4 *)(xv + at), xb = *(const float4 *)(xv + plane + at);
    float a = acc0, b = acc1;
    a = fmaf(l_bf16_lo(p.x), xa.x, a);
    b = fmaf(l_bf16_lo(q.x), xa.x, b);
    a = fmaf(l_bf16_hi(p.x), xa.y, a);
    b = fmaf(l_bf16_hi(q.x), xa.y, b);
    a = fmaf(l_bf16_lo(p.y), xa.z, a);
    b = fmaf(l_bf16_lo(q.y), xa.z, b);
    a = fmaf(l_bf16_hi(p.y), xa.w, a);
    b = fmaf(l_bf16_hi(q.y), xa.w, b);
    a = fmaf(l_bf16_lo(p.z), xb.x, a);
    b = fmaf(l_bf16_lo(q.z), xb.x, b);
    a = fmaf(l_bf16_hi(p.z), xb.y, a);
    b = fmaf(l_bf16_hi(q.z), xb.y, b);
    a = fmaf(l_bf16_lo(p.w), xb.z, a);
    b = fmaf(l_bf16_lo(q.w), xb.z, b);
    a = fmaf(l_bf16_hi(p.w), xb.w, a);
    b = fmaf(l_bf16_hi(q.w), xb.w, b);
    acc0 = k < ld ? a : acc0;
    acc1 = k < ld ? b : acc1;
}

// Choice of up to 40 experts by every wavefront for itself, an expert a lane, as l_route chooses: no barrier, no wait of one wavefront for another
// before the chosen rows can be requested.  (An expert is eight instructions.  Products behind it over those behind the workgroup's choice with two barriers
// more: up to 8 experts 0.82 of the time, 16 to 24 0.88, 32 to 40 0.97, 40 to 48 1.01, 56 to 64 1.05, 1.13 at most.)  sel: of this wavefront's own; the place
// of the lane's expert is returned.
__device__ __forceinline__ int rows_choose(float v, int E, int top, int *sel, int lane) {
    int rank = 0;
    for (int o = 0; o < E; o += 8) {
#pragma unroll
        for (int i = 0; i < 8; i++) {  // (beyond E: not larger than any, and not before any)
            const float u = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), o + i));
            rank += (u > v || (u == v && o + i < lane)) ? 1 : 0;
        }
    }
    if (lane >= E) rank = top;
    if (lane < top) sel[lane] = 0;  // (a place that no number takes, with NaN among them, stays defined)
    asm volatile("" ::: "memory");  // (a wavefront's LDS accesses are served in order)
    if (rank < top) sel[rank] = lane;
    asm volatile("" ::: "memory");
    return rank;
}
// the scores of the places, by one wavefront
__device__ __forceinline__ void rows_scores(float v, int rank, int top, int kind, float *score, int lane) {
    if (lane < top) score[lane] = 0.0f;
    asm volatile("" ::: "memory");
    if (rank < top) score[rank] = kind == LROUTE_SIGMOID_IN ? l_sigmoid(v) : v;
    asm volatile("" ::: "memory");
    if (kind != LROUTE_SOFTMAX_OUT) return;
    const float w = lane < top ? score[lane] : -INFINITY, m = wave_max_f32(w);
    const float p = lane < top ? expf(w - m) : 0.0f, sum = l_wave_sum(p);
    if (lane < top) score[lane] = p / sum;
}

// What bounds a decode step's products is the matrix bytes, so nothing may stand between the launch and the stream of loads: the
// vector is requested first, the wavefront's first step right behind it (loads return in order), and the prologue's barriers
// order LDS traffic only, so that the step stays under way while the norm is formed.  (With barriers that wait for memory, as
// __syncthreads does, 128 x 4096 rows behind a norm started streaming 6 us late.)
//
// Short launches, of which a layer's step has half a dozen, are a chain of latencies: launch (1.6 us), arguments, vector, sums, products, sums, store.  What is
// on it counts: sums by DPP, the norm's factor on the results instead of on the vector (a barrier less), whatever the prologue needs requested before
// the rows, and straight code (an instruction that is not there need not be fetched either).  Recorded launches, us, before and after: norm with pending update and
// 2566 rows of 768 3.9 -> 3.1; head norm, 768 x 768 3.7 -> 2.85, 4096 x 4096 9.9 -> 7.9; 16 rows behind a norm 3.1 -> 2.6; experts up and down at width 768
// 4.8 -> 4.2 and 4.4 -> 3.8; a side gate 3.7 -> 3.1; 134 MB behind a norm 29.1 -> 26.1.
//
// U: chunks of a row pair fetched together (2 rows x U KB per wavefront), one step.  A workgroup owns a run of row pairs and its
// wavefronts share the run's steps evenly, across the borders of pairs: with whole pairs per wavefront the rows of a 12 576 x
// 4096 matrix came to 1.5 pairs a wavefront, that is two, on 393 of 512 places.  A pair's first wavefront leaves its sums in
// s_res; wavefronts that go on with a pair leave theirs in s_part, added in order.  Four wavefronts per SIMD (128 registers): two
// workgroups a CU.
//
// V: steps of four elements a thread in which the vector is requested; Y: with a pending update.  b: the workgroup's number among the
// product's; s_mem: rows_lds() bytes.
template <int PRO, int EPI, int U, int V, bool Y>
__device__ __forceinline__ void rows_body(const RowsArgs &a, const RowsPlan &pl, int b, float *s_mem, const RowsMore &m = RowsMore(),
                                          const RowsKeys &keys = RowsKeys()) {
    __shared__ float s_red[2][ROWS_WAVES];
    __shared__ float s_part[ROWS_WAVES][2];
    __shared__ int s_head[ROWS_WAVES];  // the pair that s_part belongs to
    __shared__ int s_sel[PRO == RP_UP ? ROWS_WAVES : 1][ROWS_MAX_TOP];  // (a choice by the wavefronts, each for itself, has a row for each)
    __shared__ float s_score[ROWS_MAX_TOP];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int K = a.K, ld = a.ld, plane = pl.plane;
    const int nvec = PRO == RP_DOWN ? a.top : 1;  // vectors staged, each in its own 2 * plane floats
    float *xs = s_mem, *s_res = s_mem + nvec * 2 * plane;
    // (all that the first loads' addresses depend on is asked for at once: an argument read where it is used is a wait of its own before them)
    asm volatile("" ::"s"(pl.pairs), "s"(pl.more), "s"(pl.per_pair), "s"(pl.by_pair.mul), "s"(pl.by_pair.shift), "s"(pl.by_pair.one), "s"(a.w), "s"(a.n_rows), "s"(a.eps));
    if constexpr (PRO == RP_DOWN) asm volatile("" ::"s"(pl.by_vec.mul), "s"(pl.by_vec.shift), "s"(pl.by_vec.one), "s"(pl.per_vec), "s"(a.sel), "s"(a.rows_each));
    if constexpr (PRO == RP_UP) asm volatile("" ::"s"(pl.by_each.mul), "s"(pl.by_each.shift), "s"(pl.by_each.one), "s"(a.z), "s"(a.z_bias), "s"(a.n_experts), "s"(a.top), "s"(a.rows_each));

    // ---- the vector is requested ----------------------------------------------------------------------------------
    // (four elements a thread and step)
    const bool quads = K % 4 == 0 && (PRO != RP_HEADNORM || a.hv % 4 == 0);
    const bool fast = quads && nvec * K <= 4 * V * ROWS_THREADS;
    constexpr bool more = EPI == RE_RESID_MORE, resid = EPI == RE_RESID || more;
    constexpr bool as_is = PRO == RP_PLAIN || PRO == RP_DOWN, normed_results = PRO == RP_NORM || PRO == RP_UP;
    DecodeCtl ctl;
    if (EPI == RE_STORE_KEY && b == 0) ctl = *keys.ctl;
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr bool choice = PRO == RP_UP, chosen = PRO == RP_DOWN;  // (of experts: made here, or handed on in a.sel)
    const bool by_wave = choice && a.n_experts <= ROWS_CHOOSE;
    float z = -INFINITY, zb = 0.0f;  // an expert a lane
    int rank = 0;
    if (by_wave && lane < a.n_experts) {
        z = a.z[lane];
        if (a.z_bias) zb = a.z_bias[lane];
    }
    // (four partial sums of squares a head, and vectors of up to 4096 elements: what the head norm reads is requested with the vector, not behind the rows)
    constexpr bool heads_ahead = PRO == RP_HEADNORM && V <= 2;
    const bool sums4 = heads_ahead && a.n_split == 4;
    float4 x[V], w[as_is ? 1 : V], g[PRO == RP_HEADNORM ? V : 1], y[Y ? V : 1], yw[Y ? V : 1], sq[heads_ahead ? V : 1];
    if (Y && fast) {
#pragma unroll
        for (int u = 0; u < V; u++) {
            const int i = 4 * (t + u * ROWS_THREADS);
            y[u] = yw[u] = zero4;
            if (i < K) {
                y[u] = *(const float4 *)(a.y + i);
                yw[u] = *(const float4 *)(a.yw + i);
            }
        }
    }
    if (fast) {
#pragma unroll
        for (int u = 0; u < V; u++) {
            const int i = 4 * (t + u * ROWS_THREADS);
            x[u] = zero4;
            if (i < nvec * K) x[u] = *(const float4 *)(a.x + i);
            if constexpr (!as_is) {
                w[u] = zero4;
                if (PRO != RP_HEADNORM && i < K) w[u] = *(const float4 *)(a.normw + i);
            }
            if constexpr (PRO == RP_HEADNORM) {
                g[u] = zero4;
                if (i < K) g[u] = *(const float4 *)(a.gate + i);
            }
            if constexpr (heads_ahead) {
                sq[u] = zero4;
                if (i < K && sums4) {
                    const int h = (unsigned)i / (unsigned)a.hv;
                    sq[u] = *(const float4 *)(a.ssq + 4 * h);
                    w[u] = *(const float4 *)(a.normw + (i - h * a.hv));
                }
            }
        }
    }
    const int n_pairs = pl.pairs + (b < pl.more);
    const int64_t p0 = (int64_t)b * pl.pairs + min(b, pl.more), row0 = 2 * p0, row_end = min(2 * (p0 + n_pairs), a.n_rows);
    constexpr int kstep = U * 512;
    // (of the row whose result this thread writes first)
    float before = 0.0f;
    float plus = 0.0f, plus2 = 0.0f;
    if (resid && row0 + t < row_end) before = a.resid[row0 + t];
    if (EPI == RE_EMBED && row0 + t < row_end) before = l_bf16(a.emb[row0 + t]);
    if (more && row0 + t < row_end) {
        if (m.plus) plus = m.plus[row0 + t];
        if (m.plus2) plus2 = m.plus2[row0 + t];
    }
    asm volatile("" ::: "memory");

    // ---- the work of this wavefront: steps u0 .. u1 - 1 of the workgroup's pairs --------------------------------------
    const int total = n_pairs * pl.per_pair;
    const int u0 = (unsigned)(total * wave) / ROWS_WAVES, u1 = (unsigned)(total * (wave + 1)) / ROWS_WAVES;
    int pair = (int)rows_quot((unsigned)min(u0, total - 1), pl.by_pair), step = min(u0, total - 1) - pair * pl.per_pair;
    int v = PRO == RP_DOWN ? (int)rows_quot((unsigned)step, pl.by_vec) : 0, k = (step - v * pl.per_vec) * kstep;
    const int *sel = by_wave ? s_sel[wave] : s_sel[0];
    auto row_ptrs = [&](int pair, int v, const uint16_t *&w0, const uint16_t *&w1) {
        // (fewer than 2^31 rows, and as many in all experts together: 32 bits until the product with a row's length)
        const unsigned r = (unsigned)row0 + 2u * (unsigned)pair, r1 = r + 1 < (unsigned)row_end ? r + 1 : r, each = (unsigned)a.rows_each;
        if (PRO == RP_UP) {
            const unsigned e0 = rows_quot(r, pl.by_each), e1 = rows_quot(r1, pl.by_each);
            w0 = a.w + (uint64_t)((unsigned)sel[e0] * each + (r - e0 * each)) * (unsigned)ld;
            w1 = a.w + (uint64_t)((unsigned)sel[e1] * each + (r1 - e1 * each)) * (unsigned)ld;
        } else if (PRO == RP_DOWN) {
            const unsigned first = (unsigned)sel[v] * each;
            w0 = a.w + (uint64_t)(first + r) * (unsigned)ld;
            w1 = a.w + (uint64_t)(first + r1) * (unsigned)ld;
        } else {
            const unsigned stride = more ? (unsigned)m.stride : (unsigned)ld;
            w0 = a.w + (uint64_t)r * stride;
            w1 = a.w + (uint64_t)r1 * stride;
        }
    };
    RowsChunk cur[U], nxt[U];
    const uint16_t *w0 = nullptr, *w1 = nullptr;
    auto fetch = [&](RowsChunk (&c)[U], int k) {
#pragma unroll
        for (int u = 0; u < U; u++) rows_load(c[u], w0, w1, k + 512 * u + 8 * lane, ld);
    };
    if (chosen) {
        sel = a.sel;  // (the first step's; the others find them in LDS)
        if (t < a.top) s_sel[0][t] = sel[t];
    } else if (by_wave) {
        z += zb;
        rank = rows_choose(z, a.n_experts, a.top, s_sel[wave], lane);
    } else if (choice) {
        l_route<true>(a.z, a.z_bias, a.n_experts, a.top, a.route, s_res, s_sel[0], s_score);
    }
    row_ptrs(pair, v, w0, w1);
    fetch(cur, k);
    asm volatile("" ::: "memory");
    if (chosen) sel = s_sel[0];
    if (by_wave && wave == 0) rows_scores(z, rank, a.top, a.route, s_score, lane);
    if (choice && b == 0 && t < a.top) a.sel[t] = s_sel[0][t];  // (the first wavefront's own choice, or behind a barrier)
    if (lane == 0) s_head[wave] = -1;

    // ---- the vector -------------------------------------------------------------------------------------------
    auto put4 = [&](float *dst, int q, float4 v) { *(float4 *)(dst + (q & 1) * plane + 4 * (q >> 1)) = v; };
    auto head_scale = [&](int h) {
        float ss = 0.0f;
        for (int p = 0; p < a.n_split; p++) ss += a.ssq[h * a.n_split + p];
        return l_rsqrt(ss / (float)a.hv + a.eps);
    };
    if constexpr (normed_results) {
        if (fast) {
            if constexpr (Y) {
                float ss = 0.0f;
#pragma unroll
                for (int u = 0; u < V; u++) ss = fmaf(y[u].x, y[u].x, fmaf(y[u].y, y[u].y, fmaf(y[u].z, y[u].z, fmaf(y[u].w, y[u].w, ss))));
                const float f = a.mult * l_rsqrt(fmaf(l_block_sum_lds(ss, s_red[0]), pl.inv_K, a.eps));
#pragma unroll
                for (int u = 0; u < V; u++) {
                    const int i = 4 * (t + u * ROWS_THREADS);
                    x[u].x = fmaf(f * y[u].x, yw[u].x, x[u].x);
                    x[u].y = fmaf(f * y[u].y, yw[u].y, x[u].y);
                    x[u].z = fmaf(f * y[u].z, yw[u].z, x[u].z);
                    x[u].w = fmaf(f * y[u].w, yw[u].w, x[u].w);
                    if (b == 0 && i < K) *(float4 *)(a.x_out + i) = x[u];
                }
            }
            float ss = 0.0f;
#pragma unroll
            for (int u = 0; u < V; u++) ss = fmaf(x[u].x, x[u].x, fmaf(x[u].y, x[u].y, fmaf(x[u].z, x[u].z, fmaf(x[u].w, x[u].w, ss))));
#pragma unroll
            for (int u = 0; u < V; u++) {
                const int q = t + u * ROWS_THREADS;
                if (4 * q < ld) put4(xs, q, make_float4(x[u].x * w[u].x, x[u].y * w[u].y, x[u].z * w[u].z, x[u].w * w[u].w));
            }
            ss = l_wave_sum(ss);
            if (lane == 0) s_red[1][wave] = ss;
        } else {
            float f = 0.0f;
            if (Y) {
                float ss = 0.0f;
                for (int i = t; i < K; i += ROWS_THREADS) ss = fmaf(a.y[i], a.y[i], ss);
                f = a.mult * l_rsqrt(fmaf(l_block_sum_lds(ss, s_red[0]), pl.inv_K, a.eps));
            }
            float ss = 0.0f;
            for (int i = t; i < ld; i += ROWS_THREADS) {
                float v = 0.0f;
                if (i < K) {
                    v = a.x[i];
                    if (Y) {
                        v = fmaf(f * a.y[i], a.yw[i], v);
                        if (b == 0) a.x_out[i] = v;
                    }
                }
                ss = fmaf(v, v, ss);
                if (i < K) v *= a.normw[i];
                xs[xs_index(i, plane)] = v;
            }
            ss = l_wave_sum(ss);
            if (lane == 0) s_red[1][wave] = ss;
        }
    } else if constexpr (PRO == RP_HEADNORM) {
        auto scaled = [&](int q, float r, float4 x, float4 n, float4 g) {
            put4(xs, q, make_float4(r * x.x * n.x * g.x, r * x.y * n.y * g.y, r * x.z * n.z * g.z, r * x.w * n.w * g.w));
        };
        auto normed = [&](int q, float4 x, float4 g) {
            const int i = 4 * q;
            if (i >= ld) return;
            const int h = (unsigned)min(i, K - 4) / (unsigned)a.hv;
            if (i < K)
                scaled(q, head_scale(h), x, *(const float4 *)(a.normw + (i - h * a.hv)), g);
            else
                put4(xs, q, zero4);
        };
        if (fast && sums4) {
            if constexpr (heads_ahead) {
#pragma unroll
                for (int u = 0; u < V; u++) {
                    const int q = t + u * ROWS_THREADS;
                    const float ss = ((sq[u].x + sq[u].y) + sq[u].z) + sq[u].w;
                    if (4 * q < ld) scaled(q, l_rsqrt(ss / (float)a.hv + a.eps), x[u], w[u], g[u]);  // (zero from K on)
                }
            }
        } else if (fast) {
#pragma unroll
            for (int u = 0; u < V; u++) normed(t + u * ROWS_THREADS, x[u], g[u]);
        } else if (quads) {
            for (int q = t; 4 * q < ld; q += ROWS_THREADS)
                normed(q, 4 * q < K ? *(const float4 *)(a.x + 4 * q) : zero4, 4 * q < K ? *(const float4 *)(a.gate + 4 * q) : zero4);
        } else {
            for (int i = t; i < ld; i += ROWS_THREADS) {
                float v = 0.0f;
                if (i < K) {
                    const int h = i / a.hv;
                    v = a.x[i] * head_scale(h) * a.normw[i - h * a.hv] * a.gate[i];
                }
                xs[xs_index(i, plane)] = v;
            }
        }
    } else if (fast) {
#pragma unroll
        for (int u = 0; u < V; u++) {
            const int i = 4 * (t + u * ROWS_THREADS);
            if (i >= nvec * K) continue;
            const int v = PRO == RP_DOWN ? (unsigned)i / (unsigned)K : 0;
            put4(xs + v * 2 * plane, (i - v * K) >> 2, x[u]);
        }
        for (int i = K + t; i < ld; i += ROWS_THREADS)
            for (int v = 0; v < nvec; v++) xs[v * 2 * plane + xs_index(i, plane)] = 0.0f;
    } else if (quads) {
        for (int v = 0; v < nvec; v++)
#pragma unroll 4
            for (int q = t; 4 * q < ld; q += ROWS_THREADS) put4(xs + v * 2 * plane, q, 4 * q < K ? *(const float4 *)(a.x + (int64_t)v * K + 4 * q) : zero4);
    } else {
        for (int v = 0; v < nvec; v++)
            for (int i = t; i < ld; i += ROWS_THREADS) xs[v * 2 * plane + xs_index(i, plane)] = i < K ? a.x[(int64_t)v * K + i] : 0.0f;
    }
    l_lds_barrier();
    // (the norm's factor goes on the results: no barrier, and no sum behind one, between the vector and its products)
    float norm = 1.0f;
    if constexpr (normed_results) {
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < ROWS_WAVES; i++) ss += s_red[1][i];
        norm = l_rsqrt(fmaf(ss, pl.inv_K, a.eps));
    }

    // ---- rows -------------------------------------------------------------------------------------------------
    bool began = step == 0;  // this wavefront began the pair it is at
    float acc0 = 0.0f, acc1 = 0.0f;
    auto multiply = [&] {
        const float *xv = xs + v * 2 * plane;
#pragma unroll
        for (int i = 0; i < U; i++) rows_fma(cur[i], xv, plane, k + 512 * i + 8 * lane, ld, acc0, acc1);
    };
    auto put = [&] {
        acc0 = l_wave_sum(acc0);
        acc1 = l_wave_sum(acc1);
        if (lane == 0) {
            float *p = began ? s_res + 2 * pair : s_part[wave];
            p[0] = normed_results ? norm * acc0 : acc0;
            p[1] = normed_results ? norm * acc1 : acc1;
            if (!began) s_head[wave] = pair;
        }
    };
    // (One step by itself: behind the loop its products would begin when the last of its words is there, for the registers that the loop goes round in.
    // A matrix of 26 MB 6.8 us, 6.4 like this.)
    if (__builtin_expect(u1 - u0 == 1, 1)) {
        multiply();
        put();
    } else if (u0 < u1) {
        for (int u = u0; u + 1 < u1; u++) {
            // where the next step is; its chunks are fetched before this step's are used
            int pn = pair, vn = v, kn = k + kstep;
            if (kn >= ld) {
                kn = 0;
                if (++vn == nvec) {
                    vn = 0;
                    pn++;
                }
            }
            if (pn != pair || vn != v) row_ptrs(pn, vn, w0, w1);
            fetch(nxt, kn);
            multiply();
            if (pn != pair) {
                put();
                acc0 = acc1 = 0.0f;
                began = true;
            }
#pragma unroll
            for (int i = 0; i < U; i++) cur[i] = nxt[i];
            pair = pn;
            v = vn;
            k = kn;
        }
        multiply();
        put();
    }
    l_lds_barrier();

    // ---- results: a thread per row -------------------------------------------------------------------------------------
    unsigned long long best = 0;
    for (int i = t; row0 + i < row_end; i += ROWS_THREADS) {
        const int64_t r = row0 + i;
        const bool glu = EPI == RE_GLU || (EPI == RE_STORE_GLU && r >= a.glu_from);  // (whole pairs)
        if (glu && (i & 1)) continue;
        float val = s_res[i], up = glu ? s_res[i + 1] : 0.0f;
        if (pl.per_pair > 1) {
#pragma unroll
            for (int h = 1; h < ROWS_WAVES; h++) {
                const bool here = s_head[h] == i >> 1;
                val += here ? s_part[h][i & 1] : 0.0f;
                up += here ? s_part[h][1] : 0.0f;
            }
        }
        float f = 1.0f;
        if (PRO == RP_UP) f = s_score[rows_quot((unsigned)r, pl.by_each)];
        const float f_in = a.route == LROUTE_SIGMOID_IN ? f : 1.0f, f_out = a.route == LROUTE_SIGMOID_IN ? 1.0f : f;
        if (glu) {
            const float o = f_out * l_act(a.act, f_in * val) * (f_in * up);
            if (EPI == RE_GLU)
                a.out[r >> 1] = o;
            else
                a.out2[(r - a.glu_from) >> 1] = o;
            continue;
        }
        float o = val;
        if (resid) o = (i == t ? before : a.resid[r]) + a.mult * val;
        if (more) {
            if (m.plus) o += i == t ? plus : m.plus[r];
            if (m.plus2) o += i == t ? plus2 : m.plus2[r];
        }
        if (EPI == RE_ACT) o = l_act(a.act, val);
        if (EPI == RE_UP) o = a.route == LROUTE_SIGMOID_IN ? l_act(a.act, f * val) : f * l_act(a.act, val);
        if (EPI == RE_EMBED)
            o = l_act(a.act, val) * (i == t ? before : l_bf16(a.emb[r]));
        if (EPI == RE_STORE_AGENT)  // (read by another workgroup of the launch)
            __hip_atomic_store(a.out + r, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
            a.out[r] = o;
        if (EPI == RE_STORE_KEY) {
            const unsigned long long key = argmax_key(o, (uint32_t)r);
            best = key > best ? key : best;
        }
    }
    if constexpr (EPI == RE_STORE_KEY) {
        __shared__ unsigned long long s_best[ROWS_WAVES];
        best = wave_max_u64(best);
        if (row_end - row0 > 64) {  // (up to 64 rows are the first wavefront's)
            if (lane == 0) s_best[wave] = best;
            l_lds_barrier();
#pragma unroll
            for (int i = 0; i < ROWS_WAVES; i++) best = s_best[i] > best ? s_best[i] : best;
        }
        if (t == 0) {
            keys.keys[b] = best;
            if (b == 0) {
                ctl.picks = 1;
                *keys.next = ctl;
            }
        }
    }
}
