// Decode steps of parallel layers with latent attention (the feed-forward reads what the attention reads): the attention is a chain of
// launches that move little, the feed-forward moves most of the layer's bytes and is not needed before the chain's end.  A launch
// of either kind alone leaves HBM or the chip's latency unused, so here they share launches, workgroups of both kinds side by side:
//   k_step_pair     the queries' up projection, and from it the queries on the cached rows | the feed-forward's up product
//   k_step_latent   everything between those and the attention's output matrix | the feed-forward's down product
// Microseconds of a layer of 16 heads on a latent of 512, width 2048, at 57 to 89 positions: with experts (4 of 16, 2 x 1024 rows each) as
// launches of their own 5.2 + 4.0 + 3.8 + 7.8 + 6.5 (attention up to its output) + 11.0 + 4.4 + 7.6 = 50.3, shared 5.2 + 13.1 + 10.4 + 4.7
// = 33.4; dense of 8192 rows 48.4 and 37; a token of six layers 312 us and 248.  What bounds the shared launches is the feed-forward's
// bytes in the first (67 MB: 11 of 15.7) and the attention's latency in the second (10 to 11; alone 9 to 10).
// What the attention's part takes is the instructions and bytes of a CU, not of the chip: loads that are skipped by lanes make the
// compiler wait for all of them (19 us), v_up's rows in the matrix cores' layout, 64 bytes of sixteen rows a load, 3.4 us of address
// cycles, sums of every value over the wavefront instead of step_sum4 / step_sum16 2 us of a batch of keys.
#include "rows_dev.h"

#define SL_WAVES (ROWS_THREADS / 64)
#define SL_U (L_STEP_HEAD / SL_WAVES)  // rows of k_up, or of v_up, a wavefront: SL_U of them, sixteen
#define SL_KEYS 4                      // keys a wavefront fetches together

__device__ __forceinline__ float step_agent_load(const float *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void step_agent_store(float *p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// keys of a run: as many as keep the runs of a head at most `splits`, and no fewer than one workgroup takes in about the time that
// handing its sums over costs
__device__ __forceinline__ int step_run(int n_keys, int splits) { return max(L_STEP_RUN, ((n_keys + splits - 1) / splits + 31) & ~31); }

struct StepLds {
    float scr[SL_WAVES * L_STEP_RANK];  // parts of sums, a row per wavefront
    float m[L_STEP_SPLITS > SL_WAVES ? L_STEP_SPLITS : SL_WAVES], l[L_STEP_SPLITS > SL_WAVES ? L_STEP_SPLITS : SL_WAVES];
    float red[SL_WAVES];
    float o[L_STEP_RANK];  // the joined sum
    int last;
};
// One of n workgroups has stored its part of something (step_agent_store): true in the one that is last, which then finds all parts
// (step_agent_load).  Nobody waits for anybody; the count is zero again for the next launch.
__device__ __forceinline__ bool step_last(unsigned *count, unsigned n, int *flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the parts are in memory before the count says so)
    __syncthreads();
    if (threadIdx.x == 0) {
        const bool last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1u;
        if (last) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last;
    }
    __syncthreads();
    return *flag;
}

// One of n sums over the wavefront: lane l gets that of v[l % 4], or of v[step_sum16_of(l)].  Every step halves the sums instead of being
// taken for each of them (22 operations for four, about 60 for sixteen): a wavefront's instructions take four cycles each.
template <int CTRL>
__device__ __forceinline__ float step_swap_add(float keep, float give) {
    return keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(give), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float step_rows_sum(float c) { return l_dpp_add<0x128>(l_dpp_add<0x124>(c)); }  // row_ror:4, row_ror:8
__device__ __forceinline__ float step_sum4(const float (&v)[4], int lane) {
    const bool odd = lane & 1, high = lane & 2;
    const float a = step_swap_add<0xB1>(odd ? v[1] : v[0], odd ? v[0] : v[1]), b = step_swap_add<0xB1>(odd ? v[3] : v[2], odd ? v[2] : v[3]);
    float c = step_rows_sum(step_swap_add<0x4E>(high ? b : a, high ? a : b));
    c += __shfl_xor(c, 16, WAVE);
    return c + __shfl_xor(c, 32, WAVE);
}
__device__ __forceinline__ int step_sum16_of(int lane) { return (lane & 3) | (lane >> 4) << 2; }
__device__ __forceinline__ float step_sum16(const float (&v)[16], int lane) {
    const bool b0 = lane & 1, b1 = lane & 2, b4 = lane & 16, b5 = lane & 32;
    float a[8], b[4], c[2];
#pragma unroll
    for (int i = 0; i < 8; i++) a[i] = step_swap_add<0xB1>(b0 ? v[2 * i + 1] : v[2 * i], b0 ? v[2 * i] : v[2 * i + 1]);
#pragma unroll
    for (int i = 0; i < 4; i++) b[i] = step_rows_sum(step_swap_add<0x4E>(b1 ? a[2 * i + 1] : a[2 * i], b1 ? a[2 * i] : a[2 * i + 1]));
#pragma unroll
    for (int i = 0; i < 2; i++) c[i] = (b4 ? b[2 * i + 1] : b[2 * i]) + __shfl_xor(b4 ? b[2 * i] : b[2 * i + 1], 16, WAVE);
    return (b5 ? c[1] : c[0]) + __shfl_xor(b5 ? c[0] : c[1], 32, WAVE);
}

// A head's projected query -> its query on the cached rows: rotated, the rest through k_up^T and scaled (all of the head's 128 KB of
// k_up requested at once); head 0 also makes the token's own cache row.
__device__ __forceinline__ void step_query_body(const LatentStep &a, int h, StepLds &s) {
    const LatentShape &w = a.w;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), pos = a.ctl->pos;
    const int C = w.C, Cp = w.Cp(), Rp = w.Rp();
    const float *q = a.q + (int64_t)h * w.hq();
    float *dst = a.qa + (int64_t)h * w.ld();
    float *rot = s.scr + (SL_WAVES - 1) * L_STEP_RANK, *src = rot + L_STEP_ROT;  // (before the sums' parts go there)
    uint4 u[SL_U];  // rows wave + SL_WAVES i, 8 columns a lane
#pragma unroll
    for (int i = 0; i < SL_U; i++) {
        const int d = wave + SL_WAVES * i;
        u[i] = 8 * lane < a.ldu && d < w.D ? *(const uint4 *)(a.ukv + ((int64_t)h * w.D + d) * a.ldu + 8 * lane) : make_uint4(0, 0, 0, 0);
    }
    const int dq = wave + SL_WAVES * lane;
    const float qv = lane < SL_U && dq < w.D ? step_agent_load(q + dq) : 0.0f;
    if (wave == SL_WAVES - 1) {
        for (int i = lane; i < w.R; i += 64) src[i] = step_agent_load(q + w.D + i);
        __builtin_amdgcn_wave_barrier();
        l_rotate_norm(src, rot, w.R, w.rot, w.rot_half, a.freq, pos, 0, 0.0f, lane);
        __builtin_amdgcn_wave_barrier();
        for (int i = lane; i < Rp; i += 64) dst[Cp + i] = i < w.R ? rot[i] * w.scale : 0.0f;
    }
    if (h == 0) {
        float *row = a.cache + (int64_t)pos * w.ld();
        const float *kv = a.in + w.off_kv();
        if (wave == SL_WAVES - 2) {
            l_rotate_norm(kv + C, row + Cp, w.R, w.rot, w.rot_half, a.freq, pos, 0, 0.0f, lane);
            for (int i = w.R + lane; i < Rp; i += 64) row[Cp + i] = 0.0f;
        }
        const float v = t < C ? kv[t] : 0.0f, g = t < C ? a.kvnorm[t] : 0.0f;
        const float r = l_rsqrt(l_block_sum_lds(v * v, s.red) / (float)C + w.eps);
        if (t < Cp) row[t] = v * r * g;  // (zero from C on)
    }
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; e++) acc[e] = 0.0f;
#pragma unroll
    for (int i = 0; i < SL_U; i++) {
        const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(qv), i));
        acc[0] = fmaf(l_bf16_lo(u[i].x), x, acc[0]);
        acc[1] = fmaf(l_bf16_hi(u[i].x), x, acc[1]);
        acc[2] = fmaf(l_bf16_lo(u[i].y), x, acc[2]);
        acc[3] = fmaf(l_bf16_hi(u[i].y), x, acc[3]);
        acc[4] = fmaf(l_bf16_lo(u[i].z), x, acc[4]);
        acc[5] = fmaf(l_bf16_hi(u[i].z), x, acc[5]);
        acc[6] = fmaf(l_bf16_lo(u[i].w), x, acc[6]);
        acc[7] = fmaf(l_bf16_hi(u[i].w), x, acc[7]);
    }
    float *part = s.scr + wave * L_STEP_RANK + 8 * lane;
    *(float4 *)part = make_float4(acc[0], acc[1], acc[2], acc[3]);
    *(float4 *)(part + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
    l_lds_barrier();
    if (t < Cp) {
        float v = 0.0f;
#pragma unroll
        for (int i = 0; i < SL_WAVES; i++) v += s.scr[i * L_STEP_RANK + t];
        dst[t] = v * w.scale;
    }
}

// What the next launch's workgroups of head h will pull through one CU each is read into this XCD's L2, share j of `each`: the head's part
// of v_up, and the first keys.  (A CU pulls 52 GB/s from HBM and twice that from its L2, and v_up was 5 us of a run.)
__device__ __forceinline__ void step_warm(const LatentStep &a, int h, int j, int each) {
    const LatentShape &w = a.w;
    const uint16_t *rows = a.ukv + ((int64_t)w.H * w.D + (int64_t)h * w.V) * a.ldu;
    const int lines = (int)(((int64_t)w.V * a.ldu * 2) >> 7);  // (ldu a multiple of 64: whole lines of 128 bytes)
    const int key_lines = (int)(((int64_t)min(a.ctl->pos, L_STEP_RUN * 4) * w.ld() * 4) >> 7);
    uint32_t sink = 0;
    for (int i = j * ROWS_THREADS + threadIdx.x; i < lines + key_lines; i += each * ROWS_THREADS)
        sink |= i < lines ? *(const uint32_t *)((const char *)rows + 128 * (int64_t)i) : __float_as_uint(*(const float *)((const char *)a.cache + 128 * (int64_t)(i - lines)));
    asm volatile("" ::"v"(sink));
}

// One token's attention over the cached latent, workgroup (head, run of keys).  The wavefronts take the run's keys in turn, a key's
// row lying across the lanes, so that the row serves its score and, weighted, the sum of values from the same registers; every
// wavefront keeps a softmax of its own, and they meet in LDS.  Where a head has several runs, the workgroup that is through last joins
// them.  Then v_up, under way since the start, and the gate.
__device__ __forceinline__ void step_latent_body(const LatentStep &a, int b, StepLds &s) {
    const LatentShape &w = a.w;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int h = b % w.H, sp = b / w.H, n_keys = a.ctl->pos + 1;
    const int run = step_run(n_keys, a.splits), used = (n_keys + run - 1) / run;
    if (sp >= used) return;
    const int k0 = sp * run, k1 = min(k0 + run, n_keys);
    const int Cp = w.Cp(), Rp = w.Rp(), ld = w.ld();
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    // ---- keys k0 + wave, k0 + wave + SL_WAVES, ..: elements 4 lane .., 256 + 4 lane .. and the rotated part's element `lane` ----
    // (no load is skipped, here and below: a lane beyond the row repeats its end, and a wait can leave the later loads under way)
    const bool in0 = 4 * lane < Cp, in1 = 256 + 4 * lane < Cp, in2 = lane < Rp;
    const int at0 = min(4 * lane, Cp - 4), at1 = min(256 + 4 * lane, Cp - 4), at2 = Cp + min(lane, Rp - 1);
    struct Keys {
        float4 a[SL_KEYS], b[SL_KEYS];
        float r[SL_KEYS];
    };
    auto fetch = [&](Keys &x, int k) {
#pragma unroll
        for (int u = 0; u < SL_KEYS; u++) {
            const float *row = a.cache + (int64_t)min(k + SL_WAVES * u, k1 - 1) * ld;
            x.a[u] = *(const float4 *)(row + at0);
            x.b[u] = *(const float4 *)(row + at1);
            x.r[u] = row[at2];
        }
    };
    Keys cur;
    fetch(cur, k0 + wave);
    const float *q = a.qa + (int64_t)h * ld;
    float4 qa = *(const float4 *)(q + at0), qb = *(const float4 *)(q + at1);
    float qr = q[at2];
    // v_up: rows wave + SL_WAVES i, eight columns a lane; of the sums, lanes 0 to 3 of every sixteen keep one each.
    const int e = wave + SL_WAVES * step_sum16_of(lane);
    const float gate = a.in[w.gated ? w.off_g() + (int64_t)h * w.V + min(e, w.V - 1) : 0];
    uint4 vu[SL_U];
    auto request_values = [&](int half) {  // (in halves: the keys take the registers of one)
        const uint16_t *rows = a.ukv + ((int64_t)w.H * w.D + (int64_t)h * w.V) * a.ldu + min(8 * lane, a.ldu - 8);
#pragma unroll
        for (int i = half * SL_U / 2; i < (half + 1) * SL_U / 2; i++) vu[i] = *(const uint4 *)(rows + (int64_t)min(wave + SL_WAVES * i, w.V - 1) * a.ldu);
    };
    float mrun = -INFINITY, lrun = 0.0f;
    float4 oa = zero4, ob = zero4;
    auto pass = [&](int k) {  // keys k, k + SL_WAVES, .. in cur
        float d[SL_KEYS];
#pragma unroll
        for (int u = 0; u < SL_KEYS; u++) {
            const float4 x = cur.a[u], y = cur.b[u];
            d[u] = qr * cur.r[u];
            d[u] = fmaf(qa.x, x.x, fmaf(qa.y, x.y, fmaf(qa.z, x.z, fmaf(qa.w, x.w, d[u]))));
            d[u] = fmaf(qb.x, y.x, fmaf(qb.y, y.y, fmaf(qb.z, y.z, fmaf(qb.w, y.w, d[u]))));
        }
        // (lane l: the score of key l % 4; summed by all lanes, then chosen)
        const float sum = step_sum4(d, lane);
        const float sc = k + SL_WAVES * (lane & 3) < k1 ? sum : -INFINITY;
        float mx = fmaxf(sc, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sc), 0xB1, 0xF, 0xF, true)));
        mx = fmaxf(mx, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(mx), 0x4E, 0xF, 0xF, true)));
        // (of the first four lanes: the others' sums may differ in the last bit)
        mx = fmaxf(__int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(mx))), mrun);
        const float alpha = expf(mrun - mx), p4 = expf(sc - mx);
        mrun = mx;
        lrun *= alpha;
        oa.x *= alpha, oa.y *= alpha, oa.z *= alpha, oa.w *= alpha;
        ob.x *= alpha, ob.y *= alpha, ob.z *= alpha, ob.w *= alpha;
#pragma unroll
        for (int u = 0; u < SL_KEYS; u++) {
            if (k + SL_WAVES * u >= k1) break;
            const float p = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p4), u));
            lrun += p;
            const float4 x = cur.a[u], y = cur.b[u];
            oa.x = fmaf(p, x.x, oa.x), oa.y = fmaf(p, x.y, oa.y), oa.z = fmaf(p, x.z, oa.z), oa.w = fmaf(p, x.w, oa.w);
            ob.x = fmaf(p, y.x, ob.x), ob.y = fmaf(p, y.y, ob.y), ob.z = fmaf(p, y.z, ob.z), ob.w = fmaf(p, y.w, ob.w);
        }
    };
    auto query = [&] {  // (zero beyond the row)
        if (!in0) qa = zero4;
        if (!in1) qb = zero4;
        if (!in2) qr = 0.0f;
    };
    // (of few runs each requests v_up for itself, 128 KB that cost less than the wait of the one that is last; of many, the last alone)
    const bool ahead = used <= 4;
    if (run <= SL_WAVES * SL_KEYS) {
        if (ahead) request_values(0);
        query();
        if (k0 + wave < k1) pass(k0 + wave);
    } else {
        query();
        for (int k = k0 + wave; k < k1; k += SL_WAVES * SL_KEYS) {
            Keys nxt;
            fetch(nxt, k + SL_WAVES * SL_KEYS);
            pass(k);
            cur = nxt;
        }
        if (ahead) request_values(0);
    }
    if (ahead) request_values(1);
    // ---- the wavefronts' sums joined, then the runs' ----
    if (lane == 0) s.m[wave] = mrun, s.l[wave] = lrun;
    *(float4 *)(s.scr + wave * L_STEP_RANK + 4 * lane) = oa;
    *(float4 *)(s.scr + wave * L_STEP_RANK + 256 + 4 * lane) = ob;
    l_lds_barrier();
    float M = -INFINITY, L = 0.0f, o = 0.0f;
#pragma unroll
    for (int i = 0; i < SL_WAVES; i++) M = fmaxf(M, s.m[i]);
#pragma unroll
    for (int i = 0; i < SL_WAVES; i++) {
        const float f = s.m[i] == -INFINITY ? 0.0f : expf(s.m[i] - M);  // (a wavefront without keys)
        L = fmaf(f, s.l[i], L);
        o = fmaf(f, s.scr[i * L_STEP_RANK + t], o);
    }
    if (used > 1) {
        const int st = L_STEP_RANK + 4;
        float *p = a.part + (int64_t)h * a.splits * st, *mine = p + (int64_t)sp * st;
        step_agent_store(mine + 4 + t, o);
        if (t == 0) {
            step_agent_store(mine, M);
            step_agent_store(mine + 1, L);
        }
        if (!step_last(a.count + h, (unsigned)used, &s.last)) return;
        if (!ahead) {
            request_values(0);
            request_values(1);
        }
        if (t < used) {
            s.m[t] = step_agent_load(p + (int64_t)t * st);
            s.l[t] = step_agent_load(p + (int64_t)t * st + 1);
        }
        float x[L_STEP_SPLITS];
#pragma unroll
        for (int i = 0; i < L_STEP_SPLITS; i++) x[i] = i < used ? step_agent_load(p + (int64_t)i * st + 4 + t) : 0.0f;
        __syncthreads();
        M = -INFINITY, L = o = 0.0f;
        for (int i = 0; i < used; i++) M = fmaxf(M, s.m[i]);
#pragma unroll
        for (int i = 0; i < L_STEP_SPLITS; i++) {
            if (i >= used) break;
            const float f = expf(s.m[i] - M);
            L = fmaf(f, s.l[i], L);
            o = fmaf(f, x[i], o);
        }
    }
    // ---- v_up and the gate ----
    s.o[t] = t < Cp ? o / L : 0.0f;
    l_lds_barrier();
    {
        const float4 xa = *(const float4 *)(s.o + 8 * lane), xb = *(const float4 *)(s.o + 8 * lane + 4);
        float v[SL_U];
#pragma unroll
        for (int i = 0; i < SL_U; i++) {
            const uint4 u = vu[i];
            v[i] = l_bf16_lo(u.x) * xa.x;
            v[i] = fmaf(l_bf16_hi(u.x), xa.y, v[i]);
            v[i] = fmaf(l_bf16_lo(u.y), xa.z, v[i]);
            v[i] = fmaf(l_bf16_hi(u.y), xa.w, v[i]);
            v[i] = fmaf(l_bf16_lo(u.z), xb.x, v[i]);
            v[i] = fmaf(l_bf16_hi(u.z), xb.y, v[i]);
            v[i] = fmaf(l_bf16_lo(u.w), xb.z, v[i]);
            v[i] = fmaf(l_bf16_hi(u.w), xb.w, v[i]);
        }
        const float sum = step_sum16(v, lane);
        if ((lane & 12) == 0 && e < w.V) a.out[(int64_t)h * w.V + e] = w.gated ? sum * l_sigmoid(gate) : sum;
    }
    if (h == 0)  // (of a head's workgroups only the one that joins its runs comes here)
        for (int64_t i = (int64_t)w.H * w.V + t; i < a.cols; i += ROWS_THREADS) a.out[i] = 0.0f;
}

// workgroups below n_first: the attention; the others: rows
template <int PRO, int U>
__global__ __launch_bounds__(ROWS_THREADS, 4) void step_latent_kernel(LatentStep a, RowsArgs r, RowsPlan pl, RowsMore m, int n_first) {
    extern __shared__ __align__(16) float s_mem[];
    if ((int)blockIdx.x < n_first) {
        step_latent_body(a, blockIdx.x, *(StepLds *)s_mem);
        return;
    }
    rows_body<PRO, RE_RESID_MORE, U, 8, false>(r, pl, (int)blockIdx.x - n_first, s_mem, m);
}
// workgroups below n_first: the queries, `each` workgroups a head, of which the last takes the head's query on; the others: rows
template <int PRO, int U>
__global__ __launch_bounds__(ROWS_THREADS, 4) void step_pair_kernel(LatentStep a, RowsArgs q, RowsPlan plq, int each, RowsArgs r, RowsPlan pl, int n_first) {
    extern __shared__ __align__(16) float s_mem[];
    const int b = blockIdx.x;
    if (b >= n_first) {
        rows_body<PRO, RE_GLU, U, 2, false>(r, pl, b - n_first, s_mem);
        return;
    }
    // (a head's workgroups are those of its number among eight, as in the next launch: workgroups go to the XCDs in turn)
    const int h = b % a.w.H, j = b / a.w.H;
    rows_body<RP_NORM, RE_STORE_AGENT, 2, 2, false>(q, plq, h * each + j, s_mem);
    StepLds &s = *(StepLds *)s_mem;
    const bool last = step_last(a.count + a.w.H + h, (unsigned)each, &s.last);
    if (!last || each == 1) step_warm(a, h, each == 1 ? 0 : j, each);
    if (last) step_query_body(a, h, s);
}

// steps of 4 KB of a row where the rows are that long
static int step_u(const RowsArgs &r) { return r.ld >= 2048 ? 4 : 2; }

// workgroups that a head's rows of the query product fall to, whole pairs each: up to eight, a quarter of the chip's places in all (two, four,
// six, eight for 16 heads: a turn of 57 + 32 tokens 9.61, 9.15, 9.03, 9.05 ms)
static int step_each(const LatentShape &w, int n_cu) {
    if (w.hq() % 2 != 0) return 0;
    for (int k = 8; k >= 1; k--)
        if ((w.hq() / 2) % k == 0 && (k == 1 || w.H * k <= std::max(1, n_cu / 2))) return k;
    return 0;
}

bool k_step_fits(const LatentShape &w, int ldu, const RowsArgs &uq, const RowsArgs &up, int up_pro, const RowsArgs &down, int down_pro, int n_cu) {
    if (w.Cp() > L_STEP_RANK || ldu > L_STEP_RANK || w.D > L_STEP_HEAD || w.V > L_STEP_HEAD || w.R > L_STEP_ROT) return false;
    if (w.seq_len > (w.H < 8 ? L_STEP_KEYS / 2 : L_STEP_KEYS)) return false;
    if (uq.K > 4 * 2 * ROWS_THREADS || up.K > 4 * 2 * ROWS_THREADS) return false;  // (rows_body's V: the vector's registers)
    if (!step_each(w, n_cu) || w.H > n_cu) return false;
    // two workgroups a CU
    return rows_lds(up, up_pro, ROWS_MAX_PAIRS / 8) <= 64 * 1024 && rows_lds(down, down_pro, ROWS_MAX_PAIRS / 8) <= 64 * 1024;
}

// workgroups of a product beside n_first others: what is left of two a CU
static int64_t step_grid(const RowsArgs &r, int pro, int n_cu, int u, int n_first) {
    const int64_t n = rows_grid(r, pro, n_cu, u), pairs = (r.n_rows + 1) / 2;
    return std::max<int64_t>(std::min<int64_t>(n, 2 * (int64_t)n_cu - n_first), (pairs + ROWS_MAX_PAIRS / 8 - 2) / (ROWS_MAX_PAIRS / 8 - 1));
}

hipError_t k_step_pair(hipStream_t s, const LatentStep &a, const RowsArgs &uq, const RowsArgs &up, int pro, int n_cu) {
    const int u = step_u(up), each = step_each(a.w, n_cu);
    if (!each || uq.n_rows != (int64_t)a.w.H * a.w.hq()) return hipErrorInvalidValue;
    const int n_first = a.w.H * each;
    const RowsPlan plq = rows_plan(uq, RP_NORM, 2, n_first);
    const int64_t n = step_grid(up, pro, n_cu, u, n_first);
    const RowsPlan pl = rows_plan(up, pro, u, n);
    const size_t lds = std::max(sizeof(StepLds), std::max(rows_lds(uq, RP_NORM, plq.pairs + 1), rows_lds(up, pro, pl.pairs + 1)));
    if (lds > 64 * 1024 || up.n_rows % 2 != 0 || (pro == RP_UP && !up.sel)) return hipErrorInvalidValue;
#define GO(P, U_)                                                                                                                               \
    if (pro == P && u == U_) {                                                                                                                  \
        hipLaunchKernelGGL((step_pair_kernel<P, U_>), dim3((unsigned)(n_first + n)), dim3(ROWS_THREADS), lds, s, a, uq, plq, each, up, pl, n_first);\
        return hipGetLastError();                                                                                                               \
    }
    GO(RP_NORM, 4)
    GO(RP_NORM, 2)
    GO(RP_UP, 4)
    GO(RP_UP, 2)
#undef GO
    return hipErrorInvalidValue;
}

hipError_t k_step_latent(hipStream_t s, const LatentStep &a, const RowsArgs &down, int64_t stride, int pro, int n_cu) {
    const int u = step_u(down), n_first = a.w.H * a.splits;
    if (a.splits < 1 || a.splits > L_STEP_SPLITS) return hipErrorInvalidValue;
    const int64_t n = step_grid(down, pro, n_cu, u, std::min(a.w.H, n_cu / 2));
    const RowsPlan pl = rows_plan(down, pro, u, n);
    RowsMore m;
    m.stride = stride ? stride : down.ld;
    const size_t lds = std::max(sizeof(StepLds), rows_lds(down, pro, pl.pairs + 1));
    if (lds > 64 * 1024 || (pro == RP_DOWN && !down.sel)) return hipErrorInvalidValue;
#define GO(P, U_)                                                                                                                        \
    if (pro == P && u == U_) {                                                                                                           \
        hipLaunchKernelGGL((step_latent_kernel<P, U_>), dim3((unsigned)(n_first + n)), dim3(ROWS_THREADS), lds, s, a, down, pl, m, n_first); \
        return hipGetLastError();                                                                                                        \
    }
    GO(RP_PLAIN, 4)
    GO(RP_PLAIN, 2)
    GO(RP_DOWN, 4)
    GO(RP_DOWN, 2)
#undef GO
    return hipErrorInvalidValue;
}
