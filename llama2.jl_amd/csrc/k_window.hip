// Attention over a sliding window of the last `window` positions (the query's own included), grouped heads, interleaved
// rotation and norm of q and k, one sigmoid gate per head on the output.  Keys and values are fp32 rows of a cache that is
// linear in the position: kc[G][Dp / 4][seq_len][4], vc[G][seq_len][V].
#include "layered_dev.h"

#define WIN_MAX_HEADS 8  // query heads of a key/value head handled in one pass of the one-token kernel

// ---------------------------------------------------------------------------------------------------------------
// one token: workgroup (split of the window, key/value head).  Scores: a lane holds one key of the split, the four wavefronts
// a quarter of the key elements each.  Values: groups of threads take every so-many-th key, a thread one column.
// ---------------------------------------------------------------------------------------------------------------
// NH query heads of a key/value head at a time (a missing one has a zero query)
template <int NH>
__global__ __launch_bounds__(256) void window_step_kernel(WindowShape w, const float *freq, const float *in, float *kc, float *vc,
                                                          const DecodeCtl *ctl, float *part, float *out, int n_split) {
    extern __shared__ __align__(16) float s_mem[];
    constexpr int KA = 8, VA = 32;  // key quads and value rows a thread fetches ahead
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int g = blockIdx.y, sp = blockIdx.x, pos = ctl->pos;
    const int gq = w.H / w.G, D = w.D, Dp = w.Dp(), V = w.V, D4 = Dp / 4;
    float *s_k = s_mem, *s_q = s_k + Dp, *s_acc = s_q + NH * Dp;
    __shared__ float s_part[4][NH][L_WIN_SPLIT], s_p[NH][L_WIN_SPLIT], s_l[NH], s_m[NH];
    const int lo = max(0, pos - w.window + 1);
    const int k0 = lo + sp * L_WIN_SPLIT, n = min(L_WIN_SPLIT, pos + 1 - k0);  // this workgroup's keys
    if (n <= 0) {
        for (int i = t; i < gq; i += 256) {
            float *p = part + ((int64_t)(g * gq + i) * n_split + sp) * (V + 2);
            p[0] = -INFINITY;
            p[1] = 0.0f;
        }
        return;
    }
    const int64_t krow = (int64_t)g * D4 * w.seq_len;
    const bool has_new = k0 + n - 1 == pos;  // the token's own key and value come from its projections, not from the cache
    const int nc = has_new ? n - 1 : n;      // keys of the split that the cache holds
    const int kl = max(0, min(lane, nc - 1));  // (lanes beyond the cached keys repeat the last one)
    const int i0 = D4 * wave / 4, i1 = D4 * (wave + 1) / 4;
    const float *kp = kc + (krow + k0 + kl) * 4;
    const int tv = min(256, V), np = 256 / tv, pg = t / tv, c = t - pg * tv;  // V <= 256
    const bool mine = pg < np;
    const float *vp = vc + ((int64_t)g * w.seq_len + k0) * V + c;
    float4 kr[KA];
    float vr[VA];
#pragma unroll
    for (int u = 0; u < KA; u++) kr[u] = *(const float4 *)(kp + (int64_t)min(i0 + u, D4 - 1) * w.seq_len * 4);
#pragma unroll
    for (int u = 0; u < VA; u++) {
        const int i = pg + u * np;
        vr[u] = (mine && i < nc) ? vp[(int64_t)i * V] : 0.0f;
    }
    const float *v_new = in + w.off_v() + g * V;
    if (has_new) {
        if (wave == 3) {
            for (int i = D + lane; i < Dp; i += 64) s_k[i] = 0.0f;
            l_rotate_norm(in + w.off_k() + g * D, s_k, D, w.rot, w.rot_half, freq, pos, w.qk_norm, w.eps, lane);
        }
        for (int i = t; i < V; i += 256) vc[((int64_t)g * w.seq_len + pos) * V + i] = v_new[i];
    }
    for (int h0 = 0; h0 < gq; h0 += NH) {
        const int nh = min(NH, gq - h0);
        __syncthreads();
        for (int j = wave; j < NH; j += 4) {
            for (int i = (j < nh ? D : 0) + lane; i < Dp; i += 64) s_q[j * Dp + i] = 0.0f;
            if (j < nh) l_rotate_norm(in + (g * gq + h0 + j) * D, s_q + j * Dp, D, w.rot, w.rot_half, freq, pos, w.qk_norm, w.eps, lane);
        }
        __syncthreads();
        if (has_new && h0 == 0)
            for (int i = t; i < Dp; i += 256) kc[(krow + (int64_t)(i >> 2) * w.seq_len + pos) * 4 + (i & 3)] = s_k[i];
        float sc[NH];
#pragma unroll
        for (int j = 0; j < NH; j++) sc[j] = 0.0f;
        auto score = [&](float4 kv, int i) {
#pragma unroll
            for (int j = 0; j < NH; j++) {
                const float4 qv = *(const float4 *)(s_q + j * Dp + 4 * i);
                sc[j] = fmaf(qv.x, kv.x, sc[j]);
                sc[j] = fmaf(qv.y, kv.y, sc[j]);
                sc[j] = fmaf(qv.z, kv.z, sc[j]);
                sc[j] = fmaf(qv.w, kv.w, sc[j]);
            }
        };
#pragma unroll
        for (int u = 0; u < KA; u++)
            if (i0 + u < i1) score(kr[u], i0 + u);
        for (int i = i0 + KA; i < i1; i++) score(*(const float4 *)(kp + (int64_t)i * w.seq_len * 4), i);
#pragma unroll
        for (int j = 0; j < NH; j++) s_part[wave][j][lane] = sc[j];
        __syncthreads();
        for (int j = wave; j < nh; j += 4) {  // a wavefront per head: the whole scores, their softmax over the split
            float v = s_part[0][j][lane] + s_part[1][j][lane] + s_part[2][j][lane] + s_part[3][j][lane];
            if (has_new) {
                float own = 0.0f;
                for (int i = lane; i < D; i += 64) own = fmaf(s_q[j * Dp + i], s_k[i], own);
                own = l_wave_sum(own);
                if (lane == nc) v = own;
            }
            v = lane < n ? v * w.scale : -INFINITY;
            const float mx = wave_max_f32(v);
            const float p = lane < n ? expf(v - mx) : 0.0f;
            s_p[j][lane] = p;
            const float l = l_wave_sum(p);
            if (lane == 0) {
                s_m[j] = mx;
                s_l[j] = l;
            }
        }
        for (int j = nh + wave; j < NH; j += 4) s_p[j][lane] = 0.0f;
        __syncthreads();
        float acc[NH];
#pragma unroll
        for (int j = 0; j < NH; j++) acc[j] = 0.0f;
        if (mine) {
#pragma unroll
            for (int u = 0; u < VA; u++) {
                const int i = min(pg + u * np, L_WIN_SPLIT - 1);  // (a value past the cached keys was fetched as 0)
#pragma unroll
                for (int j = 0; j < NH; j++) acc[j] = fmaf(s_p[j][i], vr[u], acc[j]);
            }
            for (int i = pg + VA * np; i < nc; i += np) {
                const float v = vp[(int64_t)i * V];
#pragma unroll
                for (int j = 0; j < NH; j++) acc[j] = fmaf(s_p[j][i], v, acc[j]);
            }
            if (has_new && pg == 0) {
                const float v = v_new[c];
#pragma unroll
                for (int j = 0; j < NH; j++) acc[j] = fmaf(s_p[j][nc], v, acc[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < NH; j++) s_acc[j * 256 + t] = acc[j];
        __syncthreads();
        for (int idx = t; idx < nh * V; idx += 256) {
            const int j = idx / V, e = idx - j * V, h = g * gq + h0 + j;
            float v = 0.0f;
            for (int p = 0; p < np; p++) v += s_acc[j * 256 + p * tv + e];
            if (n_split == 1) {
                v /= s_l[j];
                if (w.gated) v *= l_sigmoid(in[w.off_g() + h]);
                out[h * V + e] = v;
            } else {
                float *p = part + ((int64_t)h * n_split + sp) * (V + 2);
                p[2 + e] = v;
                if (e == 0) {
                    p[0] = s_m[j];
                    p[1] = s_l[j];
                }
            }
        }
    }
}

// one workgroup per head: the splits' partial results joined
__global__ __launch_bounds__(256) void window_join_kernel(WindowShape w, const float *in, const float *part, float *out, int n_split) {
    extern __shared__ __align__(16) float s_mem[];
    float *s_f = s_mem, *s_acc = s_f + n_split;
    __shared__ float s_red[4];
    const int h = blockIdx.x, V = w.V, t = threadIdx.x, st = V + 2;
    const float *p = part + (int64_t)h * n_split * st;
    float m = -INFINITY;
    for (int i = t; i < n_split; i += 256) m = fmaxf(m, p[(int64_t)i * st]);
    m = block_max_f32(m, s_red);
    float l = 0.0f;
    for (int i = t; i < n_split; i += 256) {
        const float f = expf(p[(int64_t)i * st] - m);  // (0 for a split without keys)
        s_f[i] = f;
        l = fmaf(f, p[(int64_t)i * st + 1], l);
    }
    l = l_block_sum(l, s_red);
    const float g = (w.gated ? l_sigmoid(in[w.off_g() + h]) : 1.0f) / l;
    __syncthreads();
    const int np = 256 / V, pg = t / V, c = t - pg * V;  // V <= 256
    float v = 0.0f;
    if (pg < np)
#pragma unroll 4
        for (int i = pg; i < n_split; i += np)
            if (s_f[i] != 0.0f) v = fmaf(s_f[i], p[(int64_t)i * st + 2 + c], v);
    s_acc[t] = v;
    __syncthreads();
    if (t < V) {
        v = 0.0f;
        for (int i = 0; i < np; i++) v += s_acc[i * V + t];
        out[h * V + t] = v * g;
    }
}

hipError_t k_window_step(hipStream_t s, const WindowShape &w, const float *freq, const float *in, float *kc, float *vc,
                         const DecodeCtl *ctl, float *part, float *out) {
    const int ns = window_splits(w);
    const size_t lds = (size_t)(w.Dp() * (1 + WIN_MAX_HEADS) + WIN_MAX_HEADS * 256) * sizeof(float);
    const size_t lds_join = (size_t)(ns + 256) * sizeof(float);
    if (lds > 48 * 1024 || lds_join > 60 * 1024 || w.V > 256) return hipErrorInvalidValue;
#define GO(N) \
    hipLaunchKernelGGL((window_step_kernel<N>), dim3((unsigned)ns, (unsigned)w.G), dim3(256), lds, s, w, freq, in, kc, vc, ctl, part, out, ns)
    const int gq = w.H / w.G;
    if (gq == 1)
        GO(1);
    else if (gq == 2)
        GO(2);
    else if (gq <= 4)
        GO(4);
    else
        GO(8);
#undef GO
    if (ns > 1) hipLaunchKernelGGL(window_join_kernel, dim3((unsigned)w.H), dim3(256), lds_join, s, w, in, part, out, ns);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// many tokens
// ---------------------------------------------------------------------------------------------------------------
// one wavefront per (token, unit): units are the H query heads, then the G key/value heads
__global__ __launch_bounds__(256) void window_prepare_kernel(WindowShape w, const float *freq, const float *raw, int64_t ldr, float *kc,
                                                             float *vc, int M, int pos0, float *qf, uint16_t *qb, int hs) {
    extern __shared__ __align__(16) float s_mem[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, D = w.D;
    const int unit = blockIdx.x * 4 + wave, m = blockIdx.y, pos = pos0 + m;
    if (unit >= w.H + w.G) return;
    float *x = s_mem + wave * D;
    const float *r = raw + (int64_t)m * ldr;
    const bool isq = unit < w.H;
    const int g = unit - w.H;
    l_rotate_norm(isq ? r + unit * D : r + w.off_k() + g * D, x, D, w.rot, w.rot_half, freq, pos, w.qk_norm, w.eps, lane);
    __builtin_amdgcn_wave_barrier();
    if (isq) {
        if (qf)
            for (int i = lane; i < D; i += 64) qf[((int64_t)m * w.H + unit) * D + i] = x[i];
        if (qb)
            for (int i = lane; i < hs; i += 64) ((__bf16 *)qb)[((int64_t)m * w.H + unit) * hs + i] = (__bf16)(i < D ? x[i] : 0.0f);
        return;
    }
    for (int i = lane; i < D; i += 64) kc[(((int64_t)g * (w.Dp() / 4) + (i >> 2)) * w.seq_len + pos) * 4 + (i & 3)] = x[i];
    for (int i = lane; i < w.V; i += 64) vc[((int64_t)g * w.seq_len + pos) * w.V + i] = r[w.off_v() + g * w.V + i];
}
hipError_t k_window_prepare(hipStream_t s, const WindowShape &w, const float *freq, const float *raw, int64_t ldr, float *kc,
                            float *vc, int M, int pos0, float *qf, uint16_t *qb, int hs) {
    if (pos0 < 0 || M < 1 || pos0 + M > w.seq_len) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((w.H + w.G + 3) / 4), (unsigned)M);
    hipLaunchKernelGGL(window_prepare_kernel, grid, dim3(256), 4 * w.D * sizeof(float), s, w, freq, raw, ldr, kc, vc, M, pos0, qf, qb, hs);
    return hipGetLastError();
}

// fp32 attention on the fp32 matrix cores: workgroup = one head x 16 queries, its wavefronts take the tiles of 16 keys in turn, each with a softmax of
// its own; they join at the end.  v_mfma_f32_16x16x4_f32: lane l has A[l % 16][l / 16], B[l / 16][l % 16] and, of the result, rows
// 4 (l / 16) + r in register r, column l % 16.  Scores are keys x queries, so that a lane has four keys of one query, which is the next product's B
// operand as it stands; that product is value columns x queries, row i of its tile j being column 4 i + j of a group of 64: a lane's
// operand for four tiles is one word of 16 bytes of a key's values, and its results are 16 neighbouring columns of one query.
// What bounds it is the matrix cores' 2 x 32 cycles for every four elements of a head, on the CU whose queries see the most keys, and the loads
// ahead of them: a tile's values are requested before its scores are formed and the next tile's keys behind them.  8 heads of 128, 509 queries, all before
// them in the window: 21 us; with a key a lane and the products on the vector units 94.  Where windows are short it is the queries' loads and the
// outputs' stores, 16 bytes each a lane where sizes allow it, and wavefronts without keys, of which there are none (k_window_rows): 32 heads of 128, 2048 queries, a window of 8
// 124 us with eight wavefronts a block, 34 with one; words of 4 bytes 155.
// N: groups of 64 elements of a head (key and value elements up to 64 N); NW: wavefronts
typedef float wr_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 wr_bf16x4 __attribute__((ext_vector_type(4)));
#define WR_Q 16
template <int PREC, int N, int NW>
__global__ __launch_bounds__(64 * NW) void window_rows_kernel(WindowShape w, const float *qf, const float *raw, int64_t ldr, const float *kc,
                                                              const float *vc, int M, int pos0, void *outa, int64_t lda) {
    constexpr int DT = 4 * N;
    constexpr int NJ = NW > 1 ? NW / 2 : 1;
    __shared__ __align__(16) wr_f32x4 s_o[NJ][4 * N][64];
    __shared__ float s_m[NJ][64], s_l[NJ][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, quad = lane >> 4;
    // (the blocks that see the most keys first)
    const int h = blockIdx.y, q0 = (int)(gridDim.x - 1 - blockIdx.x) * WR_Q, D = w.D, V = w.V, D4 = w.Dp() / 4, g = h / (w.H / w.G);
    const int last = pos0 + min(q0 + WR_Q, M) - 1, first = max(0, pos0 + q0 - w.window + 1), qp = pos0 + q0 + col;
    const float *kbase = kc + (int64_t)g * D4 * w.seq_len * 4, *vbase = vc + (int64_t)g * w.seq_len * V;
    wr_f32x4 q[DT], k[DT], v[4][N], acc[N][4];
    auto fetch_keys = [&](int k0) {  // (a key that is not there repeats the last one; elements beyond the head, the head's last ones)
        const float *p = kbase + (int64_t)min(k0 + col, last) * 4;
#pragma unroll
        for (int i = 0; i < DT; i++) k[i] = *(const wr_f32x4 *)(p + (int64_t)min(4 * i + quad, D4 - 1) * w.seq_len * 4);
    };
    const bool v4 = V % 4 == 0;
    auto fetch_values = [&](int k0) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float *p = vbase + (int64_t)min(k0 + 4 * quad + r, last) * V;
#pragma unroll
            for (int n = 0; n < N; n++) {
                const int c = 64 * n + 4 * col;
                if (v4)
                    v[r][n] = *(const wr_f32x4 *)(p + min(c, V - 4));
                else
                    v[r][n] = wr_f32x4{p[min(c, V - 1)], p[min(c + 1, V - 1)], p[min(c + 2, V - 1)], p[min(c + 3, V - 1)]};
            }
        }
    };
    int k0 = first + 16 * wave;
    if (k0 <= last) fetch_keys(k0);
    {
        const float *p = qf + ((int64_t)min(q0 + col, M - 1) * w.H + h) * D;
        const bool d4 = D % 4 == 0;
#pragma unroll
        for (int i = 0; i < DT; i++) {
            const int e = 16 * i + 4 * quad;
            q[i] = d4 ? *(const wr_f32x4 *)(p + min(e, D - 4)) : wr_f32x4{p[min(e, D - 1)], p[min(e + 1, D - 1)], p[min(e + 2, D - 1)], p[min(e + 3, D - 1)]};
#pragma unroll
            for (int r = 0; r < 4; r++) q[i][r] = e + r < D ? q[i][r] : 0.0f;
        }
    }
    float mrun = -INFINITY, lrun = 0.0f;  // of query `col`: the same in the four lanes that have it
#pragma unroll
    for (int n = 0; n < N; n++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[n][j] = wr_f32x4{0.f, 0.f, 0.f, 0.f};
    for (; k0 <= last; k0 += 16 * NW) {
        fetch_values(k0);
        wr_f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
        for (int i = 0; i < DT; i++) {
            if (4 * i >= D4) break;
            const bool has = 4 * i + quad < D4;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float kr = has ? k[i][r] : 0.0f;
                if (i & 1)
                    s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kr, q[i][r], s1, 0, 0, 0);
                else
                    s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kr, q[i][r], s0, 0, 0, 0);
            }
        }
        if (k0 + 16 * NW <= last) fetch_keys(k0 + 16 * NW);
        float x[4], mx = mrun;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int key = k0 + 4 * quad + r;
            x[r] = key <= qp && qp - key < w.window && key <= last ? (s0[r] + s1[r]) * w.scale : -INFINITY;
            mx = fmaxf(mx, x[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
        const float alpha = mx == -INFINITY ? 1.0f : expf(mrun - mx);
        float sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            x[r] = x[r] == -INFINITY ? 0.0f : expf(x[r] - mx);
            sum += x[r];
        }
        mrun = mx;
        lrun = lrun * alpha + sum;  // (this lane's keys; joined at the end)
#pragma unroll
        for (int n = 0; n < N; n++) {
            if (64 * n >= V) break;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                acc[n][j] *= alpha;
#pragma unroll
                for (int r = 0; r < 4; r++) acc[n][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[r][n][j], x[r], acc[n][j], 0, 0, 0);
            }
        }
    }
    lrun += __shfl_xor(lrun, 16, WAVE);
    lrun += __shfl_xor(lrun, 32, WAVE);
    // ---- the wavefronts' sums joined, half of them onto the other half ----
#pragma unroll
    for (int half = NW / 2; half >= 1; half >>= 1) {
        if (wave >= half && wave < 2 * half) {
            s_m[wave - half][lane] = mrun;
            s_l[wave - half][lane] = lrun;
#pragma unroll
            for (int n = 0; n < N; n++)
#pragma unroll
                for (int j = 0; j < 4; j++) s_o[wave - half][4 * n + j][lane] = acc[n][j];
        }
        __syncthreads();
        if (wave < half) {
            const float mo = s_m[wave][lane], mx = fmaxf(mrun, mo);
            const float fa = mrun == -INFINITY ? 0.0f : expf(mrun - mx), fb = mo == -INFINITY ? 0.0f : expf(mo - mx);
            mrun = mx;
            lrun = lrun * fa + s_l[wave][lane] * fb;
#pragma unroll
            for (int n = 0; n < N; n++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[n][j] = acc[n][j] * fa + s_o[wave][4 * n + j][lane] * fb;
        }
        __syncthreads();
    }
    const int m = q0 + col;
    if (wave > 0 || m >= M) return;
    float f = 1.0f / lrun;
    if (w.gated) f *= l_sigmoid(raw[(int64_t)m * ldr + w.off_g() + h]);
    const int64_t at = m * lda + h * V;
#pragma unroll
    for (int n = 0; n < N; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int c = 64 * n + 16 * quad + 4 * r;
            const wr_f32x4 o = {acc[n][0][r] * f, acc[n][1][r] * f, acc[n][2][r] * f, acc[n][3][r] * f};
            if (v4) {
                if (c >= V) continue;
                if (PREC)
                    *(wr_f32x4 *)((float *)outa + at + c) = o;
                else
                    *(wr_bf16x4 *)((__bf16 *)outa + at + c) = wr_bf16x4{(__bf16)o[0], (__bf16)o[1], (__bf16)o[2], (__bf16)o[3]};
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (c + j < V) l_store_act<PREC>(outa, at + c + j, o[j]);
            }
        }
    if (h == w.H - 1)
        for (int64_t j = (int64_t)w.H * V + quad; j < lda; j += 4) l_store_act<PREC>(outa, m * lda + j, 0.0f);
}
template <int PREC, int N, int NW>
static hipError_t window_rows_go(hipStream_t s, dim3 grid, const WindowShape &w, const float *qf, const float *raw, int64_t ldr, const float *kc, const float *vc, int M,
                                 int pos0, void *outa, int64_t lda) {
    hipLaunchKernelGGL((window_rows_kernel<PREC, N, NW>), grid, dim3(64 * NW), 0, s, w, qf, raw, ldr, kc, vc, M, pos0, outa, lda);
    return hipGetLastError();
}
hipError_t k_window_rows(hipStream_t s, const WindowShape &w, const float *qf, const float *raw, int64_t ldr, const float *kc,
                         const float *vc, int M, int pos0, void *outa, int64_t lda, int prec) {
    if (w.V > 256 || w.D > 256 || pos0 < 0 || M < 1 || pos0 + M > w.seq_len) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((M + WR_Q - 1) / WR_Q), (unsigned)w.H);
    // Wavefronts a block: as many as have a tile of keys each while the chip has room for them (eight a CU; four of heads above 128 elements, which take a
    // SIMD's registers alone) or while each has six tiles; two rather than one where there is room.  Heads of 128, 2048 queries, us with one, two, four and eight
    // wavefronts: 8 heads, a window of 33 14, 15, 20, 32; of 300 51, 42, 48, 55; of 4096 274, 211, 180, 166; 2 heads, of 300 46, 26, 17, 15; 32 heads, of 33 40, 49, 63, 124.
    // 600 heads, lengths and windows: within 1.27 of the best of the four, and none slower than keys a lane on the vector units.
    const int n = (std::max(w.Dp(), w.V) + 63) / 64;
    const int64_t blocks = (int64_t)grid.x * grid.y, tiles = (std::min<int64_t>((int64_t)w.window + WR_Q - 1, pos0 + M) + 15) / 16, room = n > 2 ? 1024 : 2048;
    int nw = 2 * blocks <= room ? 2 : 1;
    for (int c : {2, 4, 8})
        if (tiles >= c && (blocks * c <= room || tiles >= 6 * c) && (c < 8 || n <= 2)) nw = c;
#define GO1(N, NW)                                                                                                                      \
    return prec ? window_rows_go<1, N, NW>(s, grid, w, qf, raw, ldr, kc, vc, M, pos0, outa, lda)                                          \
                : window_rows_go<0, N, NW>(s, grid, w, qf, raw, ldr, kc, vc, M, pos0, outa, lda)
#define GO(N)            \
    if (nw == 1)         \
        GO1(N, 1);       \
    else if (nw == 2)    \
        GO1(N, 2);       \
    else if (nw == 4)    \
        GO1(N, 4)
    if (n == 1) {
        GO(1);
        GO1(1, 8);
    } else if (n == 2) {
        GO(2);
        GO1(2, 8);
    }
    GO(4);
#undef GO1
#undef GO
    return hipErrorInvalidValue;
}
