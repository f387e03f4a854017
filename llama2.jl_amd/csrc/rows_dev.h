// One token through a bf16 matrix, the body of a workgroup (k_rows.hip has the kernels of one product, k_step.hip those of a product
// beside something else).
#pragma once

#include "layered_dev.h"
#include "rows_plan.h"

#define ROWS_MAX_EXPERTS 1024
#define ROWS_MAX_TOP 64

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
    const int at = min(k, ld - 8);
    c.p = rows_word(w0 + at);
    c.q = rows_word(w1 + at);
}
__device__ __forceinline__ void rows_fma(const RowsChunk &c, const float *xv, int plane, int k, int ld, float &acc0, float &acc1) {
    if (k >= ld) return;
    const uint4 p = c.p, q = c.q;
    const float4 xa = *(const float4 *)(xv + (k >> 1)), xb = *(const float4 *)(xv + plane + (k >> 1));
    acc0 = fmaf(l_bf16_lo(p.x), xa.x, acc0);
    acc1 = fmaf(l_bf16_lo(q.x), xa.x, acc1);
    acc0 = fmaf(l_bf16_hi(p.x), xa.y, acc0);
    acc1 = fmaf(l_bf16_hi(q.x), xa.y, acc1);
    acc0 = fmaf(l_bf16_lo(p.y), xa.z, acc0);
    acc1 = fmaf(l_bf16_lo(q.y), xa.z, acc1);
    acc0 = fmaf(l_bf16_hi(p.y), xa.w, acc0);
    acc1 = fmaf(l_bf16_hi(q.y), xa.w, acc1);
    acc0 = fmaf(l_bf16_lo(p.z), xb.x, acc0);
    acc1 = fmaf(l_bf16_lo(q.z), xb.x, acc1);
    acc0 = fmaf(l_bf16_hi(p.z), xb.y, acc0);
    acc1 = fmaf(l_bf16_hi(q.z), xb.y, acc1);
    acc0 = fmaf(l_bf16_lo(p.w), xb.z, acc0);
    acc1 = fmaf(l_bf16_lo(q.w), xb.z, acc1);
    acc0 = fmaf(l_bf16_hi(p.w), xb.w, acc0);
    acc1 = fmaf(l_bf16_hi(q.w), xb.w, acc1);
}

// What bounds a decode step's products is the matrix bytes, so nothing may stand between the launch and the stream of loads: the
// vector is requested first, the wavefront's first step right behind it (loads return in order), and the prologue's barriers
// order LDS traffic only, so that the step stays under way while the norm is formed.  (With barriers that wait for memory, as
// __syncthreads does, 128 x 4096 rows behind a norm started streaming 6 us late.)
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
    __shared__ int s_sel[ROWS_MAX_TOP];
    __shared__ float s_score[ROWS_MAX_TOP];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int K = a.K, ld = a.ld, plane = pl.plane;
    const int nvec = PRO == RP_DOWN ? a.top : 1;  // vectors staged, each in its own 2 * plane floats
    float *xs = s_mem, *s_res = s_mem + nvec * 2 * plane;

    // ---- the vector is requested ----------------------------------------------------------------------------------
    // (four elements a thread and step)
    const bool quads = K % 4 == 0 && (PRO != RP_HEADNORM || a.hv % 4 == 0);
    const bool fast = quads && nvec * K <= 4 * V * ROWS_THREADS;
    constexpr bool more = EPI == RE_RESID_MORE, resid = EPI == RE_RESID || more;
    constexpr bool as_is = PRO == RP_PLAIN || PRO == RP_DOWN;
    DecodeCtl ctl;
    if (EPI == RE_STORE_KEY && b == 0) ctl = *keys.ctl;
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 x[V], w[as_is ? 1 : V], g[PRO == RP_HEADNORM ? V : 1], y[Y ? V : 1], yw[Y ? V : 1];
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
        }
    }
    const int n_pairs = pl.pairs + (b < pl.more);
    const int64_t p0 = (int64_t)b * pl.pairs + min(b, pl.more), row0 = 2 * p0, row_end = min(2 * (p0 + n_pairs), a.n_rows);
    constexpr int kstep = U * 512;
    // (of the row whose result this thread writes first)
    float before = 0.0f;
    float plus = 0.0f, plus2 = 0.0f;
    if (resid && row0 + t < row_end) before = a.resid[row0 + t];
    if (more && row0 + t < row_end) {
        if (m.plus) plus = m.plus[row0 + t];
        if (m.plus2) plus2 = m.plus2[row0 + t];
    }
    if (EPI == RE_EMBED && row0 + t < row_end) before = l_bf16(a.emb[(int64_t)l_step_token(a.ctl, a.prompt) * a.emb_ld + row0 + t]);
    asm volatile("" ::: "memory");

    // ---- the work of this wavefront: steps u0 .. u1 - 1 of the workgroup's pairs --------------------------------------
    const int total = n_pairs * pl.per_pair;
    const int u0 = (unsigned)(total * wave) / ROWS_WAVES, u1 = (unsigned)(total * (wave + 1)) / ROWS_WAVES;
    int pair = (unsigned)min(u0, total - 1) / (unsigned)pl.per_pair, step = min(u0, total - 1) - pair * pl.per_pair;
    int v = PRO == RP_DOWN ? (unsigned)step / (unsigned)pl.per_vec : 0, k = (step - v * pl.per_vec) * kstep;
    auto row_ptrs = [&](int pair, int v, const uint16_t *&w0, const uint16_t *&w1) {
        const int64_t r = row0 + 2 * pair, r1 = r + 1 < row_end ? r + 1 : r;
        if (PRO == RP_UP) {
            const unsigned n = (unsigned)a.rows_each, e0 = (unsigned)r / n, e1 = (unsigned)r1 / n;
            w0 = a.w + ((int64_t)s_sel[e0] * a.rows_each + (r - e0 * a.rows_each)) * ld;
            w1 = a.w + ((int64_t)s_sel[e1] * a.rows_each + (r1 - e1 * a.rows_each)) * ld;
        } else if (PRO == RP_DOWN) {
            w0 = a.w + ((int64_t)s_sel[v] * a.rows_each + r) * ld;
            w1 = a.w + ((int64_t)s_sel[v] * a.rows_each + r1) * ld;
        } else {
            const int64_t stride = more ? m.stride : ld;
            w0 = a.w + r * stride;
            w1 = a.w + r1 * stride;
        }
    };
    RowsChunk cur[U], nxt[U];
    const uint16_t *w0 = nullptr, *w1 = nullptr;
    auto fetch = [&](RowsChunk (&c)[U], int k) {
#pragma unroll
        for (int u = 0; u < U; u++) rows_load(c[u], w0, w1, k + 512 * u + 8 * lane, ld);
    };
    if (PRO == RP_UP || PRO == RP_DOWN) l_route<true>(a.z, a.z_bias, a.n_experts, a.top, a.route, s_res, s_sel, s_score);
    row_ptrs(pair, v, w0, w1);
    fetch(cur, k);
    asm volatile("" ::: "memory");
    if (lane == 0) s_head[wave] = -1;

    // ---- the vector -------------------------------------------------------------------------------------------
    auto put4 = [&](float *dst, int q, float4 v) { *(float4 *)(dst + (q & 1) * plane + 4 * (q >> 1)) = v; };
    auto head_scale = [&](int h) {
        float ss = 0.0f;
        for (int p = 0; p < a.n_split; p++) ss += a.ssq[h * a.n_split + p];
        return 1.0f / sqrtf(ss / (float)a.hv + a.eps);
    };
    if constexpr (PRO == RP_NORM || PRO == RP_UP) {
        float r;
        if (fast) {
            if constexpr (Y) {
                float ss = 0.0f;
#pragma unroll
                for (int u = 0; u < V; u++) ss = fmaf(y[u].x, y[u].x, fmaf(y[u].y, y[u].y, fmaf(y[u].z, y[u].z, fmaf(y[u].w, y[u].w, ss))));
                const float f = a.mult / sqrtf(l_block_sum_lds(ss, s_red[0]) / (float)K + a.eps);
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
            r = 1.0f / sqrtf(l_block_sum_lds(ss, s_red[1]) / (float)K + a.eps);
#pragma unroll
            for (int u = 0; u < V; u++) {
                const int q = t + u * ROWS_THREADS;
                if (4 * q < ld) put4(xs, q, make_float4(r * x[u].x * w[u].x, r * x[u].y * w[u].y, r * x[u].z * w[u].z, r * x[u].w * w[u].w));
            }
        } else {
            float f = 0.0f;
            if (Y) {
                float ss = 0.0f;
                for (int i = t; i < K; i += ROWS_THREADS) ss = fmaf(a.y[i], a.y[i], ss);
                f = a.mult / sqrtf(l_block_sum_lds(ss, s_red[0]) / (float)K + a.eps);
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
            r = 1.0f / sqrtf(l_block_sum_lds(ss, s_red[1]) / (float)K + a.eps);
            for (int i = t; i < ld; i += ROWS_THREADS) xs[i] *= r;
        }
    } else if constexpr (PRO == RP_HEADNORM) {
        auto normed = [&](int q, float4 x, float4 g) {
            const int i = 4 * q;
            if (i >= ld) return;
            float4 o = zero4;
            if (i < K) {
                const int h = (unsigned)i / (unsigned)a.hv;
                const float r = head_scale(h);
                const float4 n = *(const float4 *)(a.normw + (i - h * a.hv));
                o = make_float4(r * x.x * n.x * g.x, r * x.y * n.y * g.y, r * x.z * n.z * g.z, r * x.w * n.w * g.w);
            }
            put4(xs, q, o);
        };
        if (fast) {
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
            p[0] = acc0;
            p[1] = acc1;
            if (!began) s_head[wave] = pair;
        }
    };
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
    if (u0 < u1) {
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
        if (PRO == RP_UP) f = s_score[(unsigned)r / (unsigned)a.rows_each];
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
            o = l_act(a.act, val) * (i == t ? before : l_bf16(a.emb[(int64_t)l_step_token(a.ctl, a.prompt) * a.emb_ld + r]));
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
        best = l_wave_max(best);
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
