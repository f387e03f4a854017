// Gated delta rule with one decay per head and key channel.  Per head, with state S [D][V] (fp32), unit vectors q and k,
// decay g [D], step size beta:
//   S <- diag(g) S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q = (decayed S)^T q + (k . q) u
// so both products of a token are taken of the decayed state, before its own write.
// The value columns of S are independent of one another: workgroups split them.
#include "delta_plan.h"
#include "layered_dev.h"

// ---------------------------------------------------------------------------------------------------------------
// one token: workgroup (split, head), 32 value columns x 8 groups of key channels
// ---------------------------------------------------------------------------------------------------------------
#define CONV_AHEAD 4  // taps whose inputs are fetched together

// What a channel's convolution reads: its projection, the taps' weights and the ring's slots.  No load is skipped: a weight that is not used is read all the same,
// in place of a slot that there is none for the projection again (not a slot: the token's own is being written), and both are left out of the sum.
struct DeltaConv {
    float cur, w[CONV_AHEAD], x[CONV_AHEAD];  // (x[0] is not read: it is cur)
};
__device__ __forceinline__ void delta_conv_weights(DeltaConv &v, const float *conv, const float *in, int C, int taps, int ch) {
    v.cur = in[ch];
#pragma unroll
    for (int j = 0; j < CONV_AHEAD; j++) v.w[j] = conv[(int64_t)max(taps - 1 - j, 0) * C + ch];
}
__device__ __forceinline__ void delta_conv_ring(DeltaConv &v, const float *ring, const float *in, int C, int taps, int ch, int now) {
#pragma unroll
    for (int j = 1; j < CONV_AHEAD; j++) {
        const int slot = delta_ring_slot(taps, now, j);
        const float *row = slot < 0 ? in : ring + (int64_t)slot * C;
        v.x[j] = row[ch];
    }
}
// the channel's convolution at `pos`: cur is its projection, ring slot `now` = pos % taps will hold it
__device__ __forceinline__ float delta_conv(const DeltaConv &c, const float *conv, const float *ring, int C, int taps, int ch, int pos) {
    float v = c.w[0] * c.cur;
#pragma unroll
    for (int j = 1; j < CONV_AHEAD; j++) v = j < taps && j <= pos ? fmaf(c.w[j], c.x[j], v) : v;
    for (int j = CONV_AHEAD; j < taps && j <= pos; j++)
        v = fmaf(conv[(int64_t)(taps - 1 - j) * C + ch], ring[(int64_t)((pos - j) % taps) * C + ch], v);
    return l_silu(v);
}

// 8 lanes take a bf16 row (zero-padded to ld) against a vector in LDS; every one of them gets the sum
__device__ __forceinline__ float delta_fma8(uint4 p, const float *x, float acc) {
    const float4 a = *(const float4 *)x, b = *(const float4 *)(x + 4);
    acc = fmaf(l_bf16_lo(p.x), a.x, acc);
    acc = fmaf(l_bf16_hi(p.x), a.y, acc);
    acc = fmaf(l_bf16_lo(p.y), a.z, acc);
    acc = fmaf(l_bf16_hi(p.y), a.w, acc);
    acc = fmaf(l_bf16_lo(p.z), b.x, acc);
    acc = fmaf(l_bf16_hi(p.z), b.y, acc);
    acc = fmaf(l_bf16_lo(p.w), b.z, acc);
    return fmaf(l_bf16_hi(p.w), b.w, acc);
}
__device__ __forceinline__ float delta_sum8(float acc) { return l_dpp_add<0x141>(l_dpp_add<0x4E>(l_dpp_add<0xB1>(acc))); }  // lanes l ^ 1, l ^ 2, 7 - l

// one of 16 sums over the 16 lanes of a row: lane l gets that of v[l].  Every step halves the sums: lanes l and 15 - l, l and 7 - l, l and l ^ 2, l and l ^ 1
template <int CTRL>
__device__ __forceinline__ float delta_swap_add(bool upper, float lo, float hi) {
    return (upper ? hi : lo) + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(upper ? lo : hi), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float delta_sum16(const float (&v)[16], int l) {
    float a[8], b[4], c[2];
#pragma unroll
    for (int i = 0; i < 8; i++) a[i] = delta_swap_add<0x140>(l & 8, v[i], v[i + 8]);  // row_mirror
#pragma unroll
    for (int i = 0; i < 4; i++) b[i] = delta_swap_add<0x141>(l & 4, a[i], a[i + 4]);  // row_half_mirror
#pragma unroll
    for (int i = 0; i < 2; i++) c[i] = delta_swap_add<0x4E>(l & 2, b[i], b[i + 2]);
    return delta_swap_add<0xB1>(l & 1, c[0], c[1]);
}

// What bounds this is latency: 56 KB a workgroup (1.2 us of HBM in all) in front of a chain of three sums.  So everything is
// requested at once, in the order in which it is used, no load skipped by lanes (which makes the compiler wait for all of them), and
// the barriers order LDS traffic only, so that the state is still on its way while the convolutions and decays are formed.  q and k stay as the
// convolutions leave them; what makes them unit vectors is a factor on the sums.  32 heads of 128 x 128,
// 128 workgroups: 8.1 us; with conditional loads, full barriers and rows dealt out one by one (48 LDS reads a thread where these are 12) 11.3.
// NR: rows of S per thread (D <= 8 NR)
template <int NR>
__global__ __launch_bounds__(256) void delta_step_kernel(DeltaShape d, DeltaWeights w, const float *in, float *ring, float *state,
                                                         const DecodeCtl *ctl, float *o, float *ssq, float *gate, int n_split) {
    extern __shared__ __align__(16) float s_mem[];
    float *s_q = s_mem, *s_k = s_q + 8 * NR, *s_g = s_k + 8 * NR, *s_fa = s_g + 8 * NR, *s_fg = s_fa + w.lda2;
    __shared__ float s_v[L_DELTA_COLS], s_red[2][8][L_DELTA_COLS], s_unit[3];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int sp = blockIdx.x, h = blockIdx.y, kvh = h / (d.H / d.G), pos = ctl->pos;
    const int D = d.D, V = d.V, c0 = sp * L_DELTA_COLS, GD = d.G * D, C = d.channels();
    const int col = t & 31, rg = t >> 5, c = c0 + col;
    const bool live = c < V;
    // ---- requests: convolutions, factors, state ----
    // channels t + 256 ii of the 2 D of q and k, then the workgroup's columns of v (the last one again beyond them)
    constexpr int NC = (16 * NR + L_DELTA_COLS + 255) / 256;
    const int n_ch = 2 * D + min(L_DELTA_COLS, V - c0);
    DeltaConv cv[NC];
    int ch[NC];
#pragma unroll
    for (int ii = 0; ii < NC; ii++) {
        const int i = min(t + 256 * ii, n_ch - 1), e = i >= 2 * D ? i - 2 * D : i >= D ? i - D : i;
        ch[ii] = i >= 2 * D ? 2 * GD + h * V + c0 + e : (i >= D ? GD : 0) + kvh * D + e;
        if (256 * ii + 64 * wave < n_ch) delta_conv_weights(cv[ii], w.conv, in, C, d.taps, ch[ii]);
    }
    // (the low-rank factors' inputs; longer ones in a loop below)
    float xa = 0.0f, xg = 0.0f;
    if (64 * wave < w.lda2) xa = in[d.off_a() + min(t, d.ra - 1)];
    if (64 * wave < w.ldg2) xg = in[d.off_g() + min(t, d.rg - 1)];
    const int now = pos % d.taps;
#pragma unroll
    for (int ii = 0; ii < NC; ii++)
        if (256 * ii + 64 * wave < n_ch) delta_conv_ring(cv[ii], ring, in, C, d.taps, ch[ii], now);
    // the first 128 inputs of the factors' rows
    const int l8 = t & 7, r8 = t >> 3;
    uint4 fa[NR / 4][2], fg[2];
    float bias[NR / 4];
    const float rate = w.rate[h], beta = l_sigmoid(in[d.off_b() + h]);
#pragma unroll
    for (int i = 0; i < NR / 4; i++) {
        const int64_t r = (int64_t)h * D + min(r8 + 32 * i, D - 1);
        bias[i] = w.bias[r];
#pragma unroll
        for (int e = 0; e < 2; e++) fa[i][e] = *(const uint4 *)(w.a2 + r * w.lda2 + min(8 * l8 + 64 * e, w.lda2 - 8));
    }
    const uint16_t *row_g = w.g2 + ((int64_t)h * V + min(c0 + r8, V - 1)) * w.ldg2;
#pragma unroll
    for (int e = 0; e < 2; e++) fg[e] = *(const uint4 *)(row_g + min(8 * l8 + 64 * e, w.ldg2 - 8));
    float *S = state + (int64_t)h * D * V;
    float s[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) s[i] = S[(int64_t)min(NR * rg + i, D - 1) * V + min(c, V - 1)];
    asm volatile("" ::: "memory");
    // ---- short convolutions; the token's own projections go into the ring (its slot is not read by this token) ----
    float *slot = ring + (int64_t)now * C;
#pragma unroll
    for (int ii = 0; ii < NC; ii++) {
        const int i = t + 256 * ii;
        if (256 * ii + 64 * wave >= n_ch) break;
        const float y = delta_conv(cv[ii], w.conv, ring, C, d.taps, ch[ii], pos);
        if (i < n_ch) {
            if (i >= 2 * D)
                s_v[i - 2 * D] = y;
            else if (i >= D)
                s_k[i - D] = y;
            else
                s_q[i] = y;
            if (i >= 2 * D || (sp == 0 && h % (d.H / d.G) == 0)) slot[ch[ii]] = cv[ii].cur;
        }
    }
    if (t < w.lda2) s_fa[t] = t < d.ra ? xa : 0.0f;
    if (t < w.ldg2) s_fg[t] = t < d.rg ? xg : 0.0f;
    for (int i = t + 256; i < w.lda2; i += 256) s_fa[i] = i < d.ra ? in[d.off_a() + i] : 0.0f;
    for (int i = t + 256; i < w.ldg2; i += 256) s_fg[i] = i < d.rg ? in[d.off_g() + i] : 0.0f;
    l_lds_barrier();
    // ---- what makes unit vectors of q and k, and k . q: a wavefront each ----
    if (wave < 3) {
        const float *x = wave == 0 ? s_q : s_k, *y = wave == 1 ? s_k : s_q;
        float ss = 0.0f;
        for (int e = lane; e < D; e += 64) ss = fmaf(x[e], y[e], ss);
        ss = l_wave_sum(ss);
        if (wave < 2) ss = 1.0f / sqrtf(ss + 1e-6f);
        if (wave == 0) ss *= 1.0f / sqrtf((float)D);
        if (lane == 0) s_unit[wave] = ss;
    }
    // decays of all key channels, gates of this workgroup's columns
#pragma unroll
    for (int i = 0; i < NR / 4; i++) {
        const int r = r8 + 32 * i;
        if (r >= D) break;
        const uint16_t *row = w.a2 + ((int64_t)h * D + r) * w.lda2;
        float z = 0.0f;
#pragma unroll
        for (int e = 0; e < 2; e++)
            if (8 * l8 + 64 * e < w.lda2) z = delta_fma8(fa[i][e], s_fa + 8 * l8 + 64 * e, z);
        for (int kk = 8 * l8 + 128; kk < w.lda2; kk += 64) z = delta_fma8(*(const uint4 *)(row + kk), s_fa + kk, z);
        z = delta_sum8(z) + bias[i];
        if (l8 == 0) s_g[r] = expf(-rate * l_softplus(z));
    }
    if (c0 + r8 < V) {
        float z = 0.0f;
#pragma unroll
        for (int e = 0; e < 2; e++)
            if (8 * l8 + 64 * e < w.ldg2) z = delta_fma8(fg[e], s_fg + 8 * l8 + 64 * e, z);
        for (int kk = 8 * l8 + 128; kk < w.ldg2; kk += 64) z = delta_fma8(*(const uint4 *)(row_g + kk), s_fg + kk, z);
        z = delta_sum8(z);
        if (l8 == 0) gate[h * V + c0 + r8] = l_sigmoid(z);
    }
    l_lds_barrier();
    const float uq = s_unit[0], uk = s_unit[1], kq = s_unit[2] * uq * uk;
    float dk = 0.0f, dq = 0.0f, k[NR];
#pragma unroll
    for (int i = 0; i < NR; i += 4) {
        const int r = NR * rg + i;
        const float4 g4 = *(const float4 *)(s_g + r), k4 = *(const float4 *)(s_k + r), q4 = *(const float4 *)(s_q + r);
        const float g[4] = {g4.x, g4.y, g4.z, g4.w}, q[4] = {q4.x, q4.y, q4.z, q4.w};
        k[i] = k4.x, k[i + 1] = k4.y, k[i + 2] = k4.z, k[i + 3] = k4.w;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const bool has = pos > 0 && r + j < D;  // (beyond D the words of LDS are anything)
            s[i + j] = has ? s[i + j] * g[j] : 0.0f;
            dk = has ? fmaf(s[i + j], k[i + j], dk) : dk;
            dq = has ? fmaf(s[i + j], q[j], dq) : dq;
        }
    }
    s_red[0][rg][col] = dk;
    s_red[1][rg][col] = dq;
    l_lds_barrier();
    dk = dq = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        dk += s_red[0][i][col];
        dq += s_red[1][i][col];
    }
    const float u = live ? beta * (s_v[col] - uk * dk) : 0.0f, ov = fmaf(kq, u, uq * dq), uu = uk * u;
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int r = NR * rg + i;
        if (live && r < D) S[(int64_t)r * V + c] = fmaf(k[i], uu, s[i]);
    }
    if (rg == 0) {  // (the low half of wavefront 0)
        float ss = live ? ov * ov : 0.0f;
#pragma unroll
        for (int m = 16; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, WAVE);
        if (live) o[h * V + c] = ov;
        if (col == 0) ssq[h * n_split + sp] = ss;
    }
}

hipError_t k_delta_step(hipStream_t s, const DeltaShape &d, const DeltaWeights &w, const float *in, float *ring, float *state,
                        const DecodeCtl *ctl, float *o, float *ssq, float *gate) {
    const int ns = delta_splits(d.V), nr = d.D <= 64 ? 8 : d.D <= 128 ? 16 : 32;
    if (d.D > 256) return hipErrorInvalidValue;
    const size_t lds = (size_t)(3 * 8 * nr + w.lda2 + w.ldg2) * sizeof(float);
    if (lds > 60 * 1024) return hipErrorInvalidValue;
    const dim3 grid((unsigned)ns, (unsigned)d.H);
#define GO(N) hipLaunchKernelGGL((delta_step_kernel<N>), grid, dim3(256), lds, s, d, w, in, ring, state, ctl, o, ssq, gate, ns)
    if (nr == 8)
        GO(8);
    else if (nr == 16)
        GO(16);
    else
        GO(32);
#undef GO
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// many tokens: convolutions and unit vectors.  A wavefront takes one unit (a key head's q and k, or 64 columns of a value head, or the
// rest of the row) over PREP_T consecutive tokens.  What bounds it is bytes, read and written once (the rows before a block of tokens from the L2), as
// long as every unit has all its rows under way together and a wavefront's sums do not go through LDS one by one: 16 heads of 128, 2048 tokens, 100 MB
// 32 us, against 38.
// ---------------------------------------------------------------------------------------------------------------
#define PREP_T 8

// Offsets of the CONV_AHEAD - 1 + PREP_T rows that a block of tokens reads, from row m0 - CONV_AHEAD + 1 on; rows beyond M repeat the last one.
struct PrepRows {
    int64_t at[CONV_AHEAD - 1 + PREP_T];
};
__device__ __forceinline__ float delta_raw_at(const float *raw, int64_t ldr, const float *ring, int C, int taps, int ch, int m, int pos0) {
    if (m >= 0) return raw[(int64_t)m * ldr + ch];
    const int p = pos0 + m;
    return p >= 0 ? ring[(int64_t)(p % taps) * C + ch] : 0.0f;
}
// A channel's inputs of a block of tokens, requested together
struct PrepIn {
    float x[CONV_AHEAD - 1 + PREP_T], w[CONV_AHEAD];
};
__device__ __forceinline__ void delta_conv_request(PrepIn &v, const PrepRows &rows, const float *conv, const float *raw, int64_t ldr, const float *ring, int C,
                                                   int taps, int ch, int m0, int M, int pos0) {
    if (m0 >= CONV_AHEAD - 1) {
        const float *col = raw + (int64_t)(m0 - CONV_AHEAD + 1) * ldr + ch;
        asm volatile("" : "+v"(col));  // (one address a lane: as a base a row, the compiler kept 335 scalars on the stack)
#pragma unroll
        for (int i = 0; i < CONV_AHEAD - 1 + PREP_T; i++) v.x[i] = *(const __attribute__((address_space(1))) float *)(col + rows.at[i]);
    } else {
#pragma unroll
        for (int i = 0; i < CONV_AHEAD - 1 + PREP_T; i++) {
            const int m = m0 - CONV_AHEAD + 1 + i;
            // (an input further back than the taps reach has left the ring: its weight is 0)
            v.x[i] = (m >= 0 || -m < taps) ? delta_raw_at(raw, ldr, ring, C, taps, ch, min(m, M - 1), pos0) : 0.0f;
        }
    }
#pragma unroll
    for (int j = 0; j < CONV_AHEAD; j++) v.w[j] = conv[(int64_t)max(taps - 1 - j, 0) * C + ch];
}
// the convolution and silu of a block's tokens; taps beyond CONV_AHEAD are added one by one
__device__ __forceinline__ void delta_conv_rows(const PrepIn &in, const float *conv, const float *raw, int64_t ldr, const float *ring, int C, int taps, int ch,
                                                int m0, int M, int pos0, float (&y)[PREP_T]) {
#pragma unroll
    for (int i = 0; i < PREP_T; i++) {
        float v = 0.0f;
#pragma unroll
        for (int j = 0; j < CONV_AHEAD; j++) v = j < taps ? fmaf(in.w[j], in.x[i + CONV_AHEAD - 1 - j], v) : v;
        y[i] = v;
    }
    for (int j = CONV_AHEAD; j < taps; j++) {
        const float wj = conv[(int64_t)(taps - 1 - j) * C + ch];
        for (int i = 0; i < PREP_T; i++)
            if (m0 + i < M) y[i] = fmaf(wj, delta_raw_at(raw, ldr, ring, C, taps, ch, m0 + i - j, pos0), y[i]);
    }
#pragma unroll
    for (int i = 0; i < PREP_T; i++) y[i] = l_silu(y[i]);
}
// sums over the wavefront of 16 values: lane l gets that of v[l % 16]
__device__ __forceinline__ float delta_wave_sum16(const float (&v)[16], int lane) {
    float s = delta_sum16(v, lane & 15);
    s += __shfl_xor(s, 16, WAVE);
    return s + __shfl_xor(s, 32, WAVE);
}

// NE: key channels per lane (D <= 64 NE).  TOGETHER: the inputs of all of them are requested together.  That takes 15 registers each, and pays with two of
// up to four taps; otherwise the wavefronts that it costs are worth more.  2048 tokens, 8 heads of 256 x 256, 4 and 7 taps: 31 and 65 us (together, and a token's key heads
// and values before the next token's, 34 and 98); 8 of 128 x 128, 7 and 16 taps: 34 and 98 (44 and 126).
template <int PREC, int NE, bool TOGETHER>
__global__ __launch_bounds__(256) void delta_prepare_kernel(DeltaShape d, const float *conv, const float *raw, int64_t ldr,
                                                            const float *ring, int M, int pos0, float *qkv, float *kq, float *beta,
                                                            void *fa, int64_t lfa, void *fg, int64_t lfg) {
    const int lane = threadIdx.x & 63, nv = (d.V + 63) / 64;
    // (the key heads of all tokens first: they take longest)
    const int unit = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = blockIdx.x * PREP_T, n = min(PREP_T, M - m0);
    const int C = d.channels(), GD = d.G * d.D, taps = d.taps;
    PrepRows rows;
#pragma unroll
    for (int i = 0; i < CONV_AHEAD - 1 + PREP_T; i++) rows.at[i] = min(i, M - 1 - (m0 - CONV_AHEAD + 1)) * ldr;
    if (unit > d.G + d.H * nv) return;
    if (unit == d.G + d.H * nv) {  // beta and the low-rank factors: a column of all tokens at a time
        const float *r = raw + (int64_t)m0 * ldr;
        auto column = [&](int c, float (&x)[PREP_T]) {
#pragma unroll
            for (int i = 0; i < PREP_T; i++) x[i] = r[(int64_t)min(i, n - 1) * ldr + c];
        };
        float x[PREP_T];
        for (int h = lane; h < d.H; h += 64) {
            column(d.off_b() + h, x);
#pragma unroll
            for (int i = 0; i < PREP_T; i++)
                if (i < n) beta[(int64_t)(m0 + i) * d.H + h] = l_sigmoid(x[i]);
        }
        for (int64_t j = lane; j < lfa + lfg; j += 64) {
            const bool isa = j < lfa;
            const int k = (int)(isa ? j : j - lfa), rank = isa ? d.ra : d.rg;
            column((isa ? d.off_a() : d.off_g()) + min(k, rank - 1), x);
#pragma unroll
            for (int i = 0; i < PREP_T; i++)
                if (i < n) l_store_act<PREC>(isa ? fa : fg, (int64_t)(m0 + i) * (isa ? lfa : lfg) + k, k < rank ? x[i] : 0.0f);
        }
        return;
    }
    if (unit >= d.G) {  // columns of a value head
        const int h = (unit - d.G) / nv, e = (unit - d.G - h * nv) * 64 + lane, ch = 2 * GD + h * d.V + min(e, d.V - 1);
        PrepIn in;
        float y[PREP_T];
        delta_conv_request(in, rows, conv, raw, ldr, ring, C, taps, ch, m0, M, pos0);
        delta_conv_rows(in, conv, raw, ldr, ring, C, taps, ch, m0, M, pos0, y);
        if (e < d.V)
#pragma unroll
            for (int i = 0; i < PREP_T; i++)
                if (i < n) qkv[(int64_t)(m0 + i) * C + ch] = y[i];
        return;
    }
    // a key head's q and k
    float q[NE][PREP_T], k[NE][PREP_T];
    auto channel = [&](int i) { return unit * d.D + min(lane + 64 * i, d.D - 1); };
    PrepIn in[TOGETHER ? 2 * NE : 1];
    if (TOGETHER)
#pragma unroll
        for (int i = 0; i < 2 * NE; i++) delta_conv_request(in[i], rows, conv, raw, ldr, ring, C, taps, (i & 1 ? GD : 0) + channel(i >> 1), m0, M, pos0);
#pragma unroll
    for (int i = 0; i < 2 * NE; i++) {
        PrepIn &x = in[TOGETHER ? i : 0];
        const int ch = (i & 1 ? GD : 0) + channel(i >> 1);
        if (!TOGETHER) delta_conv_request(x, rows, conv, raw, ldr, ring, C, taps, ch, m0, M, pos0);
        float(&y)[PREP_T] = i & 1 ? k[i >> 1] : q[i >> 1];
        delta_conv_rows(x, conv, raw, ldr, ring, C, taps, ch, m0, M, pos0, y);
        if (lane + 64 * (i >> 1) >= d.D)
#pragma unroll
            for (int j = 0; j < PREP_T; j++) y[j] = 0.0f;
        if (!TOGETHER) __builtin_amdgcn_sched_barrier(0);
    }
    // lane l: what makes a unit vector of token l % 8's q, or of its k (l % 16 >= 8)
    float v[2 * PREP_T], f;
#pragma unroll
    for (int j = 0; j < PREP_T; j++) {
        v[j] = v[PREP_T + j] = 0.0f;
#pragma unroll
        for (int i = 0; i < NE; i++) {
            v[j] = fmaf(q[i][j], q[i][j], v[j]);
            v[PREP_T + j] = fmaf(k[i][j], k[i][j], v[PREP_T + j]);
        }
    }
    f = 1.0f / sqrtf(delta_wave_sum16(v, lane) + 1e-6f);
    if ((lane & 15) < PREP_T) f *= 1.0f / sqrtf((float)d.D);
    float qk = 0.0f;
    if (kq) {
#pragma unroll
        for (int j = 0; j < PREP_T; j++) {
            v[j] = v[PREP_T + j] = 0.0f;
#pragma unroll
            for (int i = 0; i < NE; i++) v[j] = fmaf(q[i][j], k[i][j], v[j]);
        }
        qk = delta_wave_sum16(v, lane);
    }
#pragma unroll
    for (int j = 0; j < PREP_T; j++) {
        if (j >= n) break;
        const float rq = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), j)),
                    rk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), PREP_T + j));
        float *row = qkv + (int64_t)(m0 + j) * C + unit * d.D;
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int e = lane + 64 * i;
            if (e >= d.D) continue;
            row[e] = q[i][j] * rq;
            row[GD + e] = k[i][j] * rk;
        }
        if (kq && lane == j) kq[(int64_t)(m0 + j) * d.G + unit] = qk * rq * rk;
    }
}

hipError_t k_delta_prepare(hipStream_t s, const DeltaShape &d, const float *conv, const float *raw, int64_t ldr, const float *ring,
                           int M, int pos0, float *qkv, float *kq, float *beta, void *fa, int64_t lfa, void *fg, int64_t lfg,
                           int prec) {
    if (d.D > 256 || M < 1) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((M + PREP_T - 1) / PREP_T), (unsigned)((d.G + d.H * ((d.V + 63) / 64) + 1 + 3) / 4));
#define GO(N, TOGETHER)                                                                                                                            \
    do {                                                                                                                                           \
        if (prec)                                                                                                                                  \
            hipLaunchKernelGGL((delta_prepare_kernel<1, N, TOGETHER>), grid, dim3(256), 0, s, d, conv, raw, ldr, ring, M, pos0, qkv, kq, beta, fa, \
                               lfa, fg, lfg);                                                                                                      \
        else                                                                                                                                       \
            hipLaunchKernelGGL((delta_prepare_kernel<0, N, TOGETHER>), grid, dim3(256), 0, s, d, conv, raw, ldr, ring, M, pos0, qkv, kq, beta, fa, \
                               lfa, fg, lfg);                                                                                                      \
    } while (0)
    if (d.D <= 64)
        GO(1, true);
    else if (d.D <= 128 && d.taps <= CONV_AHEAD)
        GO(2, true);
    else if (d.D <= 128)
        GO(2, false);
    else if (d.D <= 192)
        GO(3, false);
    else
        GO(4, false);
#undef GO
    return hipGetLastError();
}

// the ring takes the last `taps` tokens' projected channels
__global__ __launch_bounds__(256) void delta_ring_kernel(const float *raw, int64_t ldr, float *ring, int C, int taps, int M, int pos0) {
    const int ch = blockIdx.x * 256 + threadIdx.x, m = M - 1 - (int)blockIdx.y;
    if (ch >= C || m < 0) return;
    ring[(int64_t)((pos0 + m) % taps) * C + ch] = raw[(int64_t)m * ldr + ch];
}
hipError_t k_delta_ring(hipStream_t s, const DeltaShape &d, const float *raw, int64_t ldr, float *ring, int M, int pos0) {
    const int C = d.channels();
    hipLaunchKernelGGL(delta_ring_kernel, dim3((unsigned)((C + 255) / 256), (unsigned)std::min(M, d.taps)), dim3(256), 0, s, raw, ldr,
                       ring, C, d.taps, M, pos0);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// the recurrence, token by token: workgroup (16 value columns, head); a wavefront holds 4 columns, 16 lanes per column,
// E = 4 NE key channels per lane (4 consecutive ones of every 64)
// ---------------------------------------------------------------------------------------------------------------
#define SCAN_T 16  // tokens staged in LDS at a time

// sum over the 16 lanes of a row, in every lane
__device__ __forceinline__ float row16_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));  // row_ror:8
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xF, 0xF, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xF, 0xF, true));
    return v;
}

template <int NE>
__global__ __launch_bounds__(256) void delta_scan_kernel(DeltaShape d, const float *qkv, const float *kq, const float *beta,
                                                         const float *lg, float *state, int M, int pos0, float *o) {
    constexpr int DP = 64 * NE;
    __shared__ __align__(16) float s_q[SCAN_T][DP], s_k[SCAN_T][DP], s_g[SCAN_T][DP];
    __shared__ float s_v[SCAN_T][16], s_o[SCAN_T][16], s_b[SCAN_T], s_kq[SCAN_T];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int h = blockIdx.y, kvh = h / (d.H / d.G), c0 = blockIdx.x * 16;
    const int D = d.D, V = d.V, C = d.channels(), GD = d.G * D;
    const int wc = 4 * wave + (lane >> 4), dl = lane & 15, c = c0 + wc;
    const bool live = c < V;
    float *S = state + (int64_t)h * D * V;
    float s[NE][4];
#pragma unroll
    for (int i = 0; i < NE; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = 64 * i + 4 * dl + j;
            s[i][j] = (live && r < D && pos0 > 0) ? S[(int64_t)r * V + c] : 0.0f;
        }
    for (int m0 = 0; m0 < M; m0 += SCAN_T) {
        const int n = min(SCAN_T, M - m0);
        __syncthreads();
        for (int i = t; i < SCAN_T * DP; i += 256) {
            const int tt = i / DP, e = i - tt * DP;
            float q = 0.0f, k = 0.0f, g = 1.0f;
            if (tt < n && e < D) {
                const float *row = qkv + (int64_t)(m0 + tt) * C + kvh * D + e;
                q = row[0];
                k = row[GD];
                g = expf(lg[(int64_t)(m0 + tt) * d.H * D + h * D + e]);
            }
            s_q[tt][e] = q;
            s_k[tt][e] = k;
            s_g[tt][e] = g;
        }
        {
            const int tt = t >> 4, e = t & 15;
            s_v[tt][e] = (tt < n && c0 + e < V) ? qkv[(int64_t)(m0 + tt) * C + 2 * GD + h * V + c0 + e] : 0.0f;
            if (e == 0) {
                s_b[tt] = tt < n ? beta[(int64_t)(m0 + tt) * d.H + h] : 0.0f;
                s_kq[tt] = tt < n ? kq[(int64_t)(m0 + tt) * d.G + kvh] : 0.0f;
            }
        }
        __syncthreads();
        for (int tt = 0; tt < n; tt++) {
            float4 k[NE], q[NE];
            float dk = 0.0f, dq = 0.0f;
#pragma unroll
            for (int i = 0; i < NE; i++) {
                const float4 g = *(const float4 *)&s_g[tt][64 * i + 4 * dl];
                k[i] = *(const float4 *)&s_k[tt][64 * i + 4 * dl];
                q[i] = *(const float4 *)&s_q[tt][64 * i + 4 * dl];
                s[i][0] *= g.x;
                s[i][1] *= g.y;
                s[i][2] *= g.z;
                s[i][3] *= g.w;
                dk = fmaf(s[i][0], k[i].x, dk);
                dq = fmaf(s[i][0], q[i].x, dq);
                dk = fmaf(s[i][1], k[i].y, dk);
                dq = fmaf(s[i][1], q[i].y, dq);
                dk = fmaf(s[i][2], k[i].z, dk);
                dq = fmaf(s[i][2], q[i].z, dq);
                dk = fmaf(s[i][3], k[i].w, dk);
                dq = fmaf(s[i][3], q[i].w, dq);
            }
            dk = row16_sum(dk);
            dq = row16_sum(dq);
            const float u = s_b[tt] * (s_v[tt][wc] - dk);
#pragma unroll
            for (int i = 0; i < NE; i++) {
                s[i][0] = fmaf(k[i].x, u, s[i][0]);
                s[i][1] = fmaf(k[i].y, u, s[i][1]);
                s[i][2] = fmaf(k[i].z, u, s[i][2]);
                s[i][3] = fmaf(k[i].w, u, s[i][3]);
            }
            if (dl == 0) s_o[tt][wc] = fmaf(s_kq[tt], u, dq);
        }
        __syncthreads();
        {
            const int tt = t >> 4, e = t & 15;
            if (tt < n && c0 + e < V) o[(int64_t)(m0 + tt) * d.H * V + h * V + c0 + e] = s_o[tt][e];
        }
    }
#pragma unroll
    for (int i = 0; i < NE; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = 64 * i + 4 * dl + j;
            if (live && r < D) S[(int64_t)r * V + c] = s[i][j];
        }
}

hipError_t k_delta_scan(hipStream_t s, const DeltaShape &d, const float *qkv, const float *kq, const float *beta, const float *lg,
                        float *state, int M, int pos0, float *o) {
    if (d.D > 256 || M < 1) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((d.V + 15) / 16), (unsigned)d.H);
#define GO(N) hipLaunchKernelGGL((delta_scan_kernel<N>), grid, dim3(256), 0, s, d, qkv, kq, beta, lg, state, M, pos0, o)
    switch ((d.D + 63) / 64) {
    case 1: GO(1); break;
    case 2: GO(2); break;
    case 3: GO(3); break;
    default: GO(4); break;
    }
#undef GO
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------------------
// the recurrence in chunks of 32 tokens, on the fp32 matrix cores.  With G_i the decays' logarithms summed over the tokens
// 0 .. i of a chunk and S0 the state before it, unrolling the recurrence gives
//   A_ij = sum_d k_i k_j exp(G_i - G_j)  (j < i),   B_ij = sum_d q_i k_j exp(G_i - G_j)  (j <= i)
//   T = (I + diag(beta) A)^-1 diag(beta),   U = T V - (T (k exp(G))) S0
//   O = (q exp(G)) S0 + B U,    S = diag(exp(G_31)) S0 + (k exp(G_31 - G))^T U
// All exponents are <= 0.  Only U and S depend on a state, so three kernels: delta_chunk_kernel makes T V and the scaled rows, for all chunks at
// once; delta_walk_kernel walks the chunks and leaves U and S0 of each; delta_out_kernel makes the outputs of all chunks at once, with the head's norm and
// gate.  What bounds the walk is its chain, 32 matrix instructions and one exchange between four wavefronts a chunk (1 us), on one CU for every 16 value
// columns; the other two, their bytes (140 and 105 MB).  16 heads of 128 x 128, 2048 tokens: 41 + 65 + 34 us, where chunks of 16 tokens, with T and the
// outputs in the walk and the norm in a launch of its own, took 39 + 126 + 13.
//
// A chunk is two tiles of 16 tokens.  Sums of logarithms are taken within a tile (E: up to a token and including it, F: behind it), so that a factor's
// exponent is never a difference of larger numbers; what lies across the tiles' border gets a tile's whole decay as a second factor.
//
// Operands are stored in the order the lanes hold them.  v_mfma_f32_16x16x4_f32: lane l has A[l % 16][l / 16], B[l / 16][l % 16]
// and, of the result, rows 4 (l / 16) + r in register r, column l % 16.  With the four steps over a tile of 16 contracted
// indexes taken as k = 4 (l / 16) + r, a result is the next product's B operand as it stands, and an A operand's four steps are
// one 16-byte word of lane l: (row l % 16; columns 4 (l / 16) .. + 3).
// ---------------------------------------------------------------------------------------------------------------
typedef float d_f32x4 __attribute__((ext_vector_type(4)));

#define WK_LD(DP_) ((DP_) + 4)  // LDS row of DP_ channels
#define WK_S 20                 // LDS row of 16 tokens
static size_t delta_chunk_lds(int DP) { return (size_t)(3 * WK_T * WK_LD(DP) + 2 * DP + 6 * 16 * WK_S + WK_T) * sizeof(float); }

__device__ __forceinline__ d_f32x4 delta_mm(const d_f32x4 a, const d_f32x4 b, d_f32x4 c) {
#pragma unroll
    for (int r = 0; r < 4; r++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
    return c;
}

template <int NW>
__global__ __launch_bounds__(256) void delta_chunk_kernel(DeltaShape d, const float *qkv, const float *beta, const float *lg, int M, float *rec) {
    constexpr int NT = 4 * NW, DP = 16 * NT, LD = WK_LD(DP);
    extern __shared__ __align__(16) float s_mem[];
    // q, k and the decays as they are; then q E, k E and k F.  s_A, s_B: the two tiles' own; s_X: A, then B, of the second against the first
    float *s_q = s_mem, *s_k = s_q + WK_T * LD, *s_g = s_k + WK_T * LD, *s_end = s_g + WK_T * LD, *s_A = s_end + 2 * DP, *s_B = s_A + 2 * 16 * WK_S,
          *s_X = s_B + 2 * 16 * WK_S, *s_b = s_X + 2 * 16 * WK_S;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), row = lane & 15, q4 = 4 * (lane >> 4);
    const int ch = blockIdx.x, h = blockIdx.y, kvh = h / (d.H / d.G), m0 = ch * WK_T, n = min(WK_T, M - m0);
    const int D = d.D, V = d.V, C = d.channels(), GD = d.G * D;
    const DeltaRec R(NT, V);
    float *out = rec + ((int64_t)ch * d.H + h) * R.floats();
    // ---- a thread takes a channel of a tile (DP 256: of both, one after the other) ----
    constexpr int NU = (2 * DP + 255) / 256;
    float l[NU][16];
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const int e = (t + 256 * u) % DP, tile = (t + 256 * u) / DP;
        if (tile > 1) break;
        const int tt0 = 16 * tile;
        float q[16], k[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {  // (no load is skipped: rows beyond M repeat the last one, channels beyond D too)
            const int64_t m = m0 + min(tt0 + i, n - 1);
            const float *r = qkv + m * C + kvh * D + min(e, D - 1);
            q[i] = r[0];
            k[i] = r[GD];
            l[u][i] = lg[(m * d.H + h) * D + min(e, D - 1)];
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const bool has = tt0 + i < n && e < D;
            l[u][i] = has ? l[u][i] : 0.0f;
            s_q[(tt0 + i) * LD + e] = has ? q[i] : 0.0f;
            s_k[(tt0 + i) * LD + e] = has ? k[i] : 0.0f;
            s_g[(tt0 + i) * LD + e] = expf(l[u][i]);
        }
    }
    if (t < WK_T) s_b[t] = t < n ? beta[(int64_t)(m0 + t) * d.H + h] : 0.0f;
    // the values of this wavefront's first tiles of columns, every fourth one
    constexpr int NV = 2;
    d_f32x4 vq[NV][2];
    auto fetch_v = [&](d_f32x4 (&x)[2], int c) {
        const float *v = qkv + (int64_t)m0 * C + 2 * GD + h * V + min(16 * c + row, V - 1);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) x[i][r] = v[(int64_t)min(16 * i + q4 + r, n - 1) * C];
    };
#pragma unroll
    for (int i = 0; i < NV; i++) fetch_v(vq[i], wave + 4 * i);
    l_lds_barrier();
    // ---- A and B of a tile: a group of 16 lanes has row j of the pairs (j, i >= j), each lane four channels of every 64; r = k_j times the
    // decays of the tokens after j.  A wavefront with early rows of one tile has late ones, which are shorter, of the other ----
#pragma unroll
    for (int tile = 0; tile < 2; tile++) {
        const int w0 = 4 * (tile ? 3 - wave : wave), j = w0 + (lane >> 4), sl = lane & 15;
        const float *tq = s_q + 16 * tile * LD, *tk = s_k + 16 * tile * LD, *tg = s_g + 16 * tile * LD;
        float a[16], b[16];
#pragma unroll
        for (int i = 0; i < 16; i++) a[i] = b[i] = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const int e = 64 * w + 4 * sl;
            d_f32x4 r = *(const d_f32x4 *)(tk + j * LD + e);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                if (i < w0) continue;  // (no row of this wavefront is that early)
                const d_f32x4 g = *(const d_f32x4 *)(tg + i * LD + e), k = *(const d_f32x4 *)(tk + i * LD + e), q = *(const d_f32x4 *)(tq + i * LD + e);
                if (i >= w0 + 4)
                    r *= g;
                else
                    r = i > j ? r * g : r;
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    a[i] = fmaf(k[c], r[c], a[i]);
                    b[i] = fmaf(q[c], r[c], b[i]);
                }
            }
        }
        const float ai = delta_sum16(a, sl), bi = delta_sum16(b, sl);  // (of pair (j, sl))
        s_A[(16 * tile + sl) * WK_S + j] = sl > j ? ai : 0.0f;
        s_B[(16 * tile + sl) * WK_S + j] = sl >= j ? bi : 0.0f;
    }
    l_lds_barrier();
    // ---- the scaled rows, in place of q, k and the decays; a thread has its own column ----
#pragma unroll
    for (int u = 0; u < NU; u++) {
        const int e = (t + 256 * u) % DP, tile = (t + 256 * u) / DP;
        if (tile > 1) break;
        float *cq = s_q + 16 * tile * LD + e, *ck = s_k + 16 * tile * LD + e, *cg = s_g + 16 * tile * LD + e;
        float sum = 0.0f;
#pragma unroll
        for (int i = 15; i >= 0; i--) {
            cg[i * LD] = ck[i * LD] * expf(sum);
            sum += l[u][i];
        }
        sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            sum += l[u][i];
            const float x = expf(sum);
            cq[i * LD] *= x;
            ck[i * LD] *= x;
        }
        s_end[tile * DP + e] = expf(sum);
    }
    l_lds_barrier();
    // ---- wavefronts 0, 1: A and B of the second tile against the first; 2, 3: a tile's T by forward substitution, a lane per column ----
    if (wave < 2) {
        const float *rows = wave ? s_q : s_k;
        d_f32x4 y[4], x;  // (in four parts, as the outputs)
#pragma unroll
        for (int i = 0; i < 4; i++) y[i] = d_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NT; i++)
            y[i & 3] = delta_mm(*(const d_f32x4 *)(rows + (16 + row) * LD + 16 * i + q4), *(const d_f32x4 *)(s_g + row * LD + 16 * i + q4), y[i & 3]);
        x = (y[0] + y[1]) + (y[2] + y[3]);
#pragma unroll
        for (int r = 0; r < 4; r++) s_X[(16 * wave + q4 + r) * WK_S + row] = x[r];
    } else if (lane < 16) {
        float *tA = s_A + 16 * (wave - 2) * WK_S;
        const float *tb = s_b + 16 * (wave - 2);
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float v = i == lane ? 1.0f : 0.0f;
#pragma unroll
            for (int j = 0; j < i; j++) v = fmaf(-tA[i * WK_S + j], x[j], v);
            x[i] = tb[i] * v;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 16; i++) tA[i * WK_S + lane] = x[i];
    }
    l_lds_barrier();
    // ---- T of the second tile against the first: -T2 A21 T1, by every wavefront for itself ----
    const d_f32x4 T1 = *(const d_f32x4 *)(s_A + row * WK_S + q4), T2 = *(const d_f32x4 *)(s_A + (16 + row) * WK_S + q4);
    {
        d_f32x4 t1, x = {0.f, 0.f, 0.f, 0.f}, y = x;
#pragma unroll
        for (int r = 0; r < 4; r++) t1[r] = s_A[(q4 + r) * WK_S + row];
        x = delta_mm(*(const d_f32x4 *)(s_X + row * WK_S + q4), t1, x);
        y = delta_mm(T2, x, y);
        l_lds_barrier();
        if (wave == 0)
#pragma unroll
            for (int r = 0; r < 4; r++) s_X[(q4 + r) * WK_S + row] = -y[r];
    }
    l_lds_barrier();
    const d_f32x4 T21 = *(const d_f32x4 *)(s_X + row * WK_S + q4);
    const d_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // ---- T V: a wavefront takes every fourth tile of columns ----
    auto put_v = [&](d_f32x4 (&x)[2], int c) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (16 * i + q4 + r >= n) x[i][r] = 0.0f;
        *(d_f32x4 *)(out + R.u(c, 0) + 4 * lane) = delta_mm(T1, x[0], zero);
        *(d_f32x4 *)(out + R.u(c, 1) + 4 * lane) = delta_mm(T2, x[1], delta_mm(T21, x[0], zero));
    };
#pragma unroll
    for (int i = 0; i < NV; i++)
        if (wave + 4 * i < R.NC) put_v(vq[i], wave + 4 * i);
    for (int c = wave + 4 * NV; c < R.NC; c += 4) {
        fetch_v(vq[0], c);
        put_v(vq[0], c);
    }
    // ---- T (k exp(G)), transposed: rows are channels; and the other scaled rows ----
#pragma unroll
    for (int ii = 0; ii < NW; ii++) {
        const int i = wave + 4 * ii, e = 16 * i + row;
        const float end0 = s_end[e], end1 = s_end[DP + e];
        d_f32x4 k0, k1, f0, f1;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            k0[r] = s_k[(q4 + r) * LD + e];
            k1[r] = s_k[(16 + q4 + r) * LD + e] * end0;
            f0[r] = s_g[(q4 + r) * LD + e] * end1;
            f1[r] = s_g[(16 + q4 + r) * LD + e];
        }
        const d_f32x4 z0 = *(const d_f32x4 *)(s_end + 16 * i + q4), q0 = *(const d_f32x4 *)(s_q + row * LD + 16 * i + q4),
                      q1 = *(const d_f32x4 *)(s_q + (16 + row) * LD + 16 * i + q4) * z0;
        *(d_f32x4 *)(out + R.kt(0, i) + 4 * lane) = delta_mm(k0, T1, zero);
        *(d_f32x4 *)(out + R.kt(1, i) + 4 * lane) = delta_mm(k1, T2, delta_mm(k0, T21, zero));
        *(d_f32x4 *)(out + R.kh(i, 0) + 4 * lane) = f0;
        *(d_f32x4 *)(out + R.kh(i, 1) + 4 * lane) = f1;
        *(d_f32x4 *)(out + R.qt(0, i) + 4 * lane) = q0;
        *(d_f32x4 *)(out + R.qt(1, i) + 4 * lane) = q1;
        if (q4 == 0) out[R.gc() + e] = e < D ? end0 * end1 : 0.0f;
    }
    if (wave < 3) *(d_f32x4 *)(out + R.b(wave) + 4 * lane) = *(const d_f32x4 *)((wave < 2 ? s_B + 16 * wave * WK_S : s_X + 16 * WK_S) + row * WK_S + q4);
}

// one chunk's operands of a wavefront with NW tiles of key channels
template <int NW>
struct DeltaOps {
    d_f32x4 kt[2][NW], kh[NW][2], gc[NW], u[2];
};

template <int NW>
__global__ __launch_bounds__(256) void delta_walk_kernel(DeltaShape d, float *rec, float *state, int M, int pos0, unsigned n_cb, unsigned n_items,
                                                         unsigned per) {
    __shared__ __align__(16) d_f32x4 s_w[2][4][2][64];
    constexpr int NT = 4 * NW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, q4 = 4 * (lane >> 4);
    // the workgroups of a head read the same records: they are dealt to one of the 8 XCDs (workgroups go to them in turn)
    const unsigned item = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (item >= n_items) return;
    const int h = (int)(item / n_cb), cb = (int)(item % n_cb), c = cb * 16 + col, D = d.D, V = d.V;
    const DeltaRec R(NT, V);
    const bool live = c < V;
    float *S = state + (int64_t)h * D * V;
    d_f32x4 s[NW];
#pragma unroll
    for (int i = 0; i < NW; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int e = 16 * (wave * NW + i) + q4 + r;
            s[i][r] = (live && e < D && pos0 > 0) ? S[(int64_t)e * V + c] : 0.0f;
        }
    const int n_ch = (M + WK_T - 1) / WK_T;
    // wavefront-uniform base and this lane's fixed offset from it
    float *rec_h = rec + (int64_t)h * R.floats();
    const int64_t rec_step = (int64_t)d.H * R.floats();
    const unsigned l4 = 4u * lane;
    // request `at` of a chunk's kt and T V (the first 2 NW + 2), and of its kh and gc (3 NW)
    auto fetch_kt = [&](DeltaOps<NW> &x, int ch, int at) {
        const float *p = rec_h + min(ch, n_ch - 1) * rec_step + l4;
        if (at < 2 * NW)
            x.kt[at & 1][at >> 1] = *(const d_f32x4 *)(p + R.kt(at & 1, wave * NW + (at >> 1)));
        else
            x.u[at - 2 * NW] = *(const d_f32x4 *)(p + R.u(cb, at - 2 * NW));
    };
    auto fetch_kh = [&](DeltaOps<NW> &x, int ch, int at) {
        const float *p = rec_h + min(ch, n_ch - 1) * rec_step;
        if (at < 2 * NW)
            x.kh[at >> 1][at & 1] = *(const d_f32x4 *)(p + R.kh(wave * NW + (at >> 1), at & 1) + l4);
        else
            x.gc[at - 2 * NW] = *(const d_f32x4 *)(p + R.gc() + 16 * (wave * NW + at - 2 * NW) + q4);
    };
    // Chunk ch, whose operands x holds; meanwhile the rest of chunk ch + 2 is requested (into y), then, as x comes free, the first part of ch + 3.  The requests
    // stand between the matrix instructions one by one (a wavefront that issues a chunk's twelve in a row waits until the memory pipeline has taken
    // them: 71 us against 65), and none is left out, so that how many are under way is known when the code is compiled
    // (a wait is one for all of them otherwise: 86 us).
    auto walk = [&](DeltaOps<NW> &x, DeltaOps<NW> &y, int ch) {
        const int b = ch & 1;
        float *p = rec_h + ch * rec_step + l4;
        const d_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        d_f32x4 w0 = zero, w1 = zero;
#pragma unroll
        for (int j = 0; j < 4 * NW; j++) {
            w0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[0][j >> 2][j & 3], s[j >> 2][j & 3], w0, 0, 0, 0);
            w1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[1][j >> 2][j & 3], s[j >> 2][j & 3], w1, 0, 0, 0);
            if (j < 3 * NW)
                fetch_kh(y, ch + 2, j);
            else
                *(d_f32x4 *)(p + R.s0(cb, wave * NW + j - 3 * NW)) = s[j - 3 * NW];
            __builtin_amdgcn_sched_barrier(0);
        }
        // (the first wavefront takes T V off its part, behind its products, and its part is added last: sums of small numbers round less)
        s_w[b][wave][0][lane] = wave ? w0 : w0 - x.u[0];
        s_w[b][wave][1][lane] = wave ? w1 : w1 - x.u[1];
#pragma unroll
        for (int i = 0; i < NW; i++) s[i] *= x.gc[i];
        // LDS writes done, then the barrier; what is under way to and from memory is not waited for
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const d_f32x4 u0 = -(s_w[b][1][0][lane] + s_w[b][2][0][lane] + s_w[b][3][0][lane] + s_w[b][0][0][lane]);
        const d_f32x4 u1 = -(s_w[b][1][1][lane] + s_w[b][2][1][lane] + s_w[b][3][1][lane] + s_w[b][0][1][lane]);
        constexpr int n_kt = 2 * NW + 2;
#pragma unroll
        for (int j = 0; j < 8; j++) {
#pragma unroll
            for (int i = 0; i < NW; i++)
                s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kh[i][j >> 2][j & 3], j < 4 ? u0[j & 3] : u1[j & 3], s[i], 0, 0, 0);
#pragma unroll
            for (int at = j * n_kt / 8; at < (j + 1) * n_kt / 8; at++) fetch_kt(x, ch + 3, at);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (wave < 2) *(d_f32x4 *)(p + R.u(cb, wave)) = wave ? u1 : u0;
    };
    // (U takes the place of T V, which the first wavefront alone uses, before the barrier behind which U is written)
    DeltaOps<NW> x0, x1, x2;
    auto first = [&](DeltaOps<NW> &x, int ch, bool all) {
#pragma unroll
        for (int at = 0; at < 2 * NW + 2; at++) fetch_kt(x, ch, at);
#pragma unroll
        for (int at = 0; at < 3 * NW; at++)
            if (all) fetch_kh(x, ch, at);
        __builtin_amdgcn_sched_barrier(0);
    };
    first(x0, 0, true);
    first(x1, 1, true);
    first(x2, 2, false);
    int ch = 0;  // (n_ch is the same for every wavefront: so is every barrier)
    for (; ch + 3 <= n_ch; ch += 3) {
        walk(x0, x2, ch);
        walk(x1, x0, ch + 1);
        walk(x2, x1, ch + 2);
    }
    if (ch < n_ch) walk(x0, x2, ch);
    if (ch + 1 < n_ch) walk(x1, x0, ch + 1);
#pragma unroll
    for (int i = 0; i < NW; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int e = 16 * (wave * NW + i) + q4 + r;
            if (live && e < D) S[(int64_t)e * V + c] = s[i][r];
        }
}

// outputs of a (chunk, head), normed over the head and gated: a wavefront takes every fourth tile of value columns
template <int PREC, int NW>
__global__ __launch_bounds__(256) void delta_out_kernel(DeltaShape d, const float *rec, const float *gate, const float *normw, int M, void *outa, int64_t lda) {
    constexpr int NT = 4 * NW, LO = 256 + 4;
    __shared__ float s_o[WK_T * LO], s_ss[4][WK_T];
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), col = lane & 15, q4 = 4 * (lane >> 4);
    const int ch = blockIdx.x, h = blockIdx.y, m0 = ch * WK_T, n = min(WK_T, M - m0), V = d.V, HV = d.H * V;
    const DeltaRec R(NT, V);
    const float *p = rec + ((int64_t)ch * d.H + h) * R.floats() + 4 * lane;
    const d_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // gates of the wavefront's rows wave + 4 i (requested behind the operands)
    constexpr int RW = WK_T / 4, NG = 2;
    const float *gp = gate + (int64_t)m0 * HV + h * V;
    float g[NG][RW], nw[NG];
    auto fetch_gates = [&](float (&x)[RW], float &w, int j) {
#pragma unroll
        for (int i = 0; i < RW; i++) x[i] = gp[(int64_t)min(wave + 4 * i, n - 1) * HV + min(j, V - 1)];
        w = normw[min(j, V - 1)];
    };
    float ss[2][4];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) ss[i][r] = 0.0f;
    if (wave < R.NC) {
        d_f32x4 qt[2][NT], s0[NT], u0, u1;
        auto fetch = [&](int c) {
#pragma unroll
            for (int i = 0; i < NT; i++) s0[i] = *(const d_f32x4 *)(p + R.s0(c, i));
            u0 = *(const d_f32x4 *)(p + R.u(c, 0));
            u1 = *(const d_f32x4 *)(p + R.u(c, 1));
        };
        fetch(wave);
#pragma unroll
        for (int i = 0; i < NT; i++) {
            qt[0][i] = *(const d_f32x4 *)(p + R.qt(0, i));
            qt[1][i] = *(const d_f32x4 *)(p + R.qt(1, i));
        }
        const d_f32x4 B1 = *(const d_f32x4 *)(p + R.b(0)), B2 = *(const d_f32x4 *)(p + R.b(1)), B21 = *(const d_f32x4 *)(p + R.b(2));
#pragma unroll
        for (int k = 0; k < NG; k++) fetch_gates(g[k], nw[k], 64 * k + lane);
        for (int c = wave; c < R.NC; c += 4) {
            d_f32x4 z[2];  // (long sums in four parts: they round less, and a part's next step finds its last one done)
#pragma unroll
            for (int k = 0; k < 2; k++) {
                d_f32x4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0, p2 = p0, p3 = p0;
#pragma unroll
                for (int i = 0; i < NT; i += 2)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        if (i < NT / 2)
                            p0 = __builtin_amdgcn_mfma_f32_16x16x4f32(qt[k][i][r], s0[i][r], p0, 0, 0, 0);
                        else
                            p2 = __builtin_amdgcn_mfma_f32_16x16x4f32(qt[k][i][r], s0[i][r], p2, 0, 0, 0);
                        if (i < NT / 2)
                            p1 = __builtin_amdgcn_mfma_f32_16x16x4f32(qt[k][i + 1][r], s0[i + 1][r], p1, 0, 0, 0);
                        else
                            p3 = __builtin_amdgcn_mfma_f32_16x16x4f32(qt[k][i + 1][r], s0[i + 1][r], p3, 0, 0, 0);
                    }
                z[k] = (p0 + p1) + (p2 + p3);
            }
            const d_f32x4 y0 = z[0] + delta_mm(B1, u0, zero), y1 = z[1] + delta_mm(B2, u1, delta_mm(B21, u0, zero));
            if (c + 4 < R.NC) fetch(c + 4);
            const int at = 16 * c + col;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                s_o[(q4 + r) * LO + at] = y0[r];
                s_o[(16 + q4 + r) * LO + at] = y1[r];
                if (at < V) {
                    ss[0][r] = fmaf(y0[r], y0[r], ss[0][r]);
                    ss[1][r] = fmaf(y1[r], y1[r], ss[1][r]);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float v = row16_sum(ss[i][r]);
            if (col == 0) s_ss[wave][16 * i + q4 + r] = v;
        }
    l_lds_barrier();
    if (wave >= R.NC)
#pragma unroll
        for (int k = 0; k < NG; k++) fetch_gates(g[k], nw[k], 64 * k + lane);
    float rms[RW];
#pragma unroll
    for (int i = 0; i < RW; i++) {
        const int at = wave + 4 * i;
        rms[i] = 1.0f / sqrtf((s_ss[0][at] + s_ss[1][at] + s_ss[2][at] + s_ss[3][at]) / (float)V + d.eps);
    }
    auto put = [&](const float (&x)[RW], float w, int j) {
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const int at = wave + 4 * i;
            if (at < n && j < V) l_store_act<PREC>(outa, (int64_t)(m0 + at) * lda + h * V + j, s_o[at * LO + j] * rms[i] * w * x[i]);
        }
    };
#pragma unroll
    for (int k = 0; k < NG; k++) put(g[k], nw[k], 64 * k + lane);
    for (int j = 64 * NG + lane; j < V; j += 64) {
        fetch_gates(g[0], nw[0], j);
        put(g[0], nw[0], j);
    }
    if (h == d.H - 1)
        for (int i = wave; i < n; i += 4)
            for (int64_t j = (int64_t)HV + lane; j < lda; j += 64) l_store_act<PREC>(outa, (int64_t)(m0 + i) * lda + j, 0.0f);
}

template <int NW>
static hipError_t delta_walk_launch(hipStream_t s, const DeltaShape &d, const float *qkv, const float *beta, const float *lg, float *state, int M, int pos0,
                                    float *rec, const float *gate, const float *normw, void *outa, int64_t lda, int prec) {
    const dim3 g1((unsigned)((M + WK_T - 1) / WK_T), (unsigned)d.H);
    const unsigned n_cb = (unsigned)((d.V + 15) / 16), n_items = n_cb * (unsigned)d.H, per = (n_items + 7) / 8;
    const size_t lds = delta_chunk_lds(64 * NW);
    if (lds > 60 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void *)delta_chunk_kernel<NW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((delta_chunk_kernel<NW>), g1, dim3(256), lds, s, d, qkv, beta, lg, M, rec);
    hipLaunchKernelGGL((delta_walk_kernel<NW>), dim3(8 * per), dim3(256), 0, s, d, rec, state, M, pos0, n_cb, n_items, per);
    if (prec)
        hipLaunchKernelGGL((delta_out_kernel<1, NW>), g1, dim3(256), 0, s, d, rec, gate, normw, M, outa, lda);
    else
        hipLaunchKernelGGL((delta_out_kernel<0, NW>), g1, dim3(256), 0, s, d, rec, gate, normw, M, outa, lda);
    return hipGetLastError();
}
// ---------------------------------------------------------------------------------------------------------------
// the same in chunks of 16 tokens, where delta_plan.h says so: the walk makes the outputs too,
//   U = T (V - (k exp(G)) S0),   O = (q exp(G)) S0 + B U,   S = diag(exp(G_15)) S0 + (k exp(G_15 - G))^T U
// and no state goes to memory but the last.  delta_chunk16_kernel makes the scaled rows, T and B, and the head norm is a launch of its own.
//
// the record of one (chunk, head), NT tiles of 16 key channels (a multiple of 4): kt, qt, kh: [NT][64][4]; T, B: [64][4]; exp(G_15): [16 NT]
// ---------------------------------------------------------------------------------------------------------------
#define CH_T DELTA_CHUNK16

template <int NW>
__global__ __launch_bounds__(256) void delta_chunk16_kernel(DeltaShape d, const float *qkv, const float *beta, const float *lg, int M,
                                                          float *rec) {
    constexpr int NT = 4 * NW, DP = 16 * NT;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // s_g: the decays, then their logarithms' sums
    __shared__ __align__(16) float s_q[CH_T * DP], s_k[CH_T * DP], s_g[CH_T * DP];
    __shared__ float s_A[CH_T][CH_T + 1], s_B[CH_T][CH_T + 1], s_T[CH_T][CH_T + 1], s_b[CH_T];
    const int ch = blockIdx.x, h = blockIdx.y, kvh = h / (d.H / d.G), m0 = ch * CH_T, n = min(CH_T, M - m0);
    const int D = d.D, C = d.channels(), GD = d.G * D;
    // a thread has one column of 16 / (256 / columns) rows at a time: column e, rows r0, r0 + RS, ...
    constexpr int CB = DP < 256 ? DP : 256, RS = 256 / CB, NR = CH_T / RS;  // (DP: 64, 128, 192 or 256)
    const int e0 = t % CB, r0 = t / CB;
    float l[NR];
    if (r0 < RS) {
        float q[NR], k[NR];
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const int tt = r0 + RS * i;
            q[i] = k[i] = l[i] = 0.0f;
            if (tt < n && e0 < D) {
                const float *row = qkv + (int64_t)(m0 + tt) * C + kvh * D + e0;
                q[i] = row[0];
                k[i] = row[GD];
                l[i] = lg[((int64_t)(m0 + tt) * d.H + h) * D + e0];
            }
        }
#pragma unroll
        for (int i = 0; i < NR; i++) {
            const int at = (r0 + RS * i) * DP + e0;
            s_q[at] = q[i];
            s_k[at] = k[i];
            s_g[at] = expf(l[i]);
        }
    }
    if (t < CH_T) s_b[t] = t < n ? beta[(int64_t)(m0 + t) * d.H + h] : 0.0f;
    __syncthreads();
    // A and B: a group of 16 lanes has row j of the pairs (j, i > j), each lane every 16th channel; r = k_j times the decays of
    // the tokens after j
    {
        const int j = 4 * wave + (lane >> 4), sl = lane & 15;
        float a[CH_T], b[CH_T];
#pragma unroll
        for (int i = 0; i < CH_T; i++) a[i] = b[i] = 0.0f;
        for (int e = sl; e < D; e += 16) {
            float r = s_k[j * DP + e];
#pragma unroll
            for (int i = 0; i < CH_T; i++) {
                if (i > j) r *= s_g[i * DP + e];
                const float u = i >= j ? r : 0.0f;
                a[i] = fmaf(s_k[i * DP + e], u, a[i]);
                b[i] = fmaf(s_q[i * DP + e], u, b[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < CH_T; i++) {
            a[i] = row16_sum(a[i]);
            b[i] = row16_sum(b[i]);
            if (sl == i) {
                s_A[i][j] = i > j ? a[i] : 0.0f;
                s_B[i][j] = b[i];
            }
        }
    }
    __syncthreads();
    // T by forward substitution, a lane per column
    if (t < CH_T) {
        float x[CH_T];
#pragma unroll
        for (int i = 0; i < CH_T; i++) {
            float v = i == t ? 1.0f : 0.0f;
#pragma unroll
            for (int j = 0; j < i; j++) v = fmaf(-s_A[i][j], x[j], v);
            x[i] = s_b[i] * v;
            s_T[i][t] = x[i];
        }
    }
    // sums of the logarithms, in place of the decays (whose readers are done)
    if (r0 < RS)
#pragma unroll
        for (int i = 0; i < NR; i++) s_g[(r0 + RS * i) * DP + e0] = l[i];
    __syncthreads();
    for (int e = t; e < DP; e += 256) {
        float g = 0.0f;
#pragma unroll
        for (int i = 0; i < CH_T; i++) {
            g += s_g[i * DP + e];
            s_g[i * DP + e] = g;
        }
    }
    __syncthreads();
    float *out = rec + ((int64_t)ch * d.H + h) * delta_rec16_floats(NT);
    for (int idx = t; idx < NT * 64; idx += 256) {
        const int tile = idx >> 6, l = idx & 63, row = l & 15, q4 = 4 * (l >> 4);
        float4 kt, qt, kh;
        {
            const int o = row * DP + 16 * tile + q4;
            const float4 k = *(const float4 *)(s_k + o), q = *(const float4 *)(s_q + o), G = *(const float4 *)(s_g + o);
            const float4 x = make_float4(expf(G.x), expf(G.y), expf(G.z), expf(G.w));
            kt = make_float4(k.x * x.x, k.y * x.y, k.z * x.z, k.w * x.w);
            qt = make_float4(q.x * x.x, q.y * x.y, q.z * x.z, q.w * x.w);
        }
        {  // row: the channel, columns: tokens
            const int e = 16 * tile + row;
            const float Gc = s_g[15 * DP + e];
            kh = make_float4(s_k[q4 * DP + e] * expf(Gc - s_g[q4 * DP + e]), s_k[(q4 + 1) * DP + e] * expf(Gc - s_g[(q4 + 1) * DP + e]),
                             s_k[(q4 + 2) * DP + e] * expf(Gc - s_g[(q4 + 2) * DP + e]),
                             s_k[(q4 + 3) * DP + e] * expf(Gc - s_g[(q4 + 3) * DP + e]));
        }
        *(float4 *)(out + 4 * idx) = kt;
        *(float4 *)(out + 256 * NT + 4 * idx) = qt;
        *(float4 *)(out + 512 * NT + 4 * idx) = kh;
    }
    if (t < 128) {
        const float(*m)[CH_T + 1] = wave ? s_B : s_T;
        const int row = lane & 15, q4 = 4 * (lane >> 4);
        *(float4 *)(out + 768 * NT + 256 * wave + 4 * lane) = make_float4(m[row][q4], m[row][q4 + 1], m[row][q4 + 2], m[row][q4 + 3]);
    }
    for (int e = t; e < DP; e += 256) out[768 * NT + 512 + e] = e < D ? expf(s_g[15 * DP + e]) : 0.0f;
}

// one chunk's operands of a wavefront with NW tiles of key channels
template <int NW>
struct DeltaOps16 {
    d_f32x4 kt[NW], qt[NW], kh[NW], gc[NW], T;
    float B, v[4];
};

// (records, rows of v and rows of o exist for whole chunks: what a sequence's last chunk has beyond it counts as zero)
template <int NW>
__global__ __launch_bounds__(256) void delta_walk16_kernel(DeltaShape d, const float *rec, const float *qkv, float *state, int M, int pos0,
                                                         float *o, unsigned n_cb, unsigned n_items, unsigned per) {
    __shared__ __align__(16) d_f32x4 s_w[2][4][64];
    __shared__ float s_o[2][4][4][64];
    constexpr int NT = 4 * NW;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 15, q4 = 4 * (lane >> 4);
    // the workgroups of a head read the same records: they are dealt to one of the 8 XCDs (workgroups go to them in turn)
    const unsigned item = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (item >= n_items) return;
    const int h = (int)(item / n_cb), c = (int)(item % n_cb) * 16 + col, D = d.D, V = d.V, C = d.channels(), HV = d.H * V;
    const bool live = c < V;
    float *S = state + (int64_t)h * D * V;
    d_f32x4 s[NW];
#pragma unroll
    for (int i = 0; i < NW; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int e = 16 * (wave * NW + i) + q4 + r;
            s[i][r] = (live && e < D && pos0 > 0) ? S[(int64_t)e * V + c] : 0.0f;
        }
    const int n_ch = (M + CH_T - 1) / CH_T;
    // wavefront-uniform bases and this lane's fixed offsets from them
    const float *rec_h = rec + (int64_t)h * delta_rec16_floats(NT) + 256 * (wave * NW);
    const int64_t rec_step = (int64_t)d.H * delta_rec16_floats(NT);
    const float *v_h = qkv + 2 * d.G * D + h * V;
    float *o_h = o + (int64_t)wave * HV + h * V;
    const unsigned l4 = 4u * lane, ov = (unsigned)(q4 * HV + c);
    unsigned vv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) vv[r] = (unsigned)((q4 + r) * C + (live ? c : 0));
    auto fetch = [&](DeltaOps16<NW> &x, int ch) {
        const float *p = rec_h + ch * rec_step;
#pragma unroll
        for (int i = 0; i < NW; i++) {
            x.kt[i] = *(const d_f32x4 *)(p + 256 * i + l4);
            x.qt[i] = *(const d_f32x4 *)(p + 256 * (NT + i) + l4);
            x.kh[i] = *(const d_f32x4 *)(p + 256 * (2 * NT + i) + l4);
        }
        p -= 256 * (wave * NW);
#pragma unroll
        for (int i = 0; i < NW; i++) x.gc[i] = *(const d_f32x4 *)(p + 768 * NT + 512 + 16 * (wave * NW + i) + q4);
        x.T = *(const d_f32x4 *)(p + 768 * NT + l4);
        x.B = (p + wave)[768 * NT + 256 + l4];
        const float *v = v_h + (int64_t)ch * CH_T * C;
#pragma unroll
        for (int r = 0; r < 4; r++) x.v[r] = v[vv[r]];
    };
    // the output row 4 (lane / 16) + wave of a chunk, from the four wavefronts' parts
    auto put = [&](int ch) {
        const int b = ch & 1;
        const float y = s_o[b][wave][0][lane] + s_o[b][wave][1][lane] + s_o[b][wave][2][lane] + s_o[b][wave][3][lane];
        if (live) (o_h + (int64_t)ch * CH_T * HV)[ov] = y;
    };
    auto walk = [&](DeltaOps16<NW> &x, int ch) {
        const int b = ch & 1;
        d_f32x4 w = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NW; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) w = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kt[i][r], s[i][r], w, 0, 0, 0);
        s_w[b][wave][lane] = w;
#pragma unroll
        for (int i = 0; i < NW; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) y = __builtin_amdgcn_mfma_f32_16x16x4f32(x.qt[i][r], s[i][r], y, 0, 0, 0);
        // LDS writes done, then the barrier (which also says that the parts of the previous chunk's output are all there);
        // the operands under way from memory are not waited for
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        w = s_w[b][0][lane] + s_w[b][1][lane] + s_w[b][2][lane] + s_w[b][3][lane];
        d_f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; r++) u = __builtin_amdgcn_mfma_f32_16x16x4f32(x.T[r], (ch * CH_T + q4 + r < M ? x.v[r] : 0.0f) - w[r], u, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < NW; i++) {
            s[i] *= x.gc[i];
#pragma unroll
            for (int r = 0; r < 4; r++) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kh[i][r], u[r], s[i], 0, 0, 0);
        }
        // B U: this wavefront's quarter of the contracted tokens
        const float uw = wave == 0 ? u[0] : wave == 1 ? u[1] : wave == 2 ? u[2] : u[3];
        y = __builtin_amdgcn_mfma_f32_16x16x4f32(x.B, uw, y, 0, 0, 0);
        if (ch) put(ch - 1);
#pragma unroll
        for (int r = 0; r < 4; r++) s_o[b][r][wave][lane] = y[r];
    };
    // the operands of three chunks are held or under way
    DeltaOps16<NW> x0, x1, x2;
    fetch(x0, 0);
    fetch(x1, min(1, n_ch - 1));
    fetch(x2, min(2, n_ch - 1));
    for (int ch = 0; ch < n_ch; ch += 3) {  // (n_ch is the same for every wavefront: so is every barrier)
        walk(x0, ch);
        fetch(x0, min(ch + 3, n_ch - 1));
        if (ch + 1 >= n_ch) break;
        walk(x1, ch + 1);
        fetch(x1, min(ch + 4, n_ch - 1));
        if (ch + 2 >= n_ch) break;
        walk(x2, ch + 2);
        fetch(x2, min(ch + 5, n_ch - 1));
    }
    __syncthreads();
    put(n_ch - 1);
#pragma unroll
    for (int i = 0; i < NW; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int e = 16 * (wave * NW + i) + q4 + r;
            if (live && e < D) S[(int64_t)e * V + c] = s[i][r];
        }
}

template <int NW>
static hipError_t delta_walk16_launch(hipStream_t s, const DeltaShape &d, const float *qkv, const float *beta, const float *lg, float *state, int M, int pos0,
                                      float *rec, float *o) {
    const dim3 g1((unsigned)((M + CH_T - 1) / CH_T), (unsigned)d.H);
    const unsigned n_cb = (unsigned)((d.V + 15) / 16), n_items = n_cb * (unsigned)d.H, per = (n_items + 7) / 8;
    hipLaunchKernelGGL((delta_chunk16_kernel<NW>), g1, dim3(256), 0, s, d, qkv, beta, lg, M, rec);
    hipLaunchKernelGGL((delta_walk16_kernel<NW>), dim3(8 * per), dim3(256), 0, s, d, rec, qkv, state, M, pos0, o, n_cb, n_items, per);
    return hipGetLastError();
}

hipError_t k_delta_walk(hipStream_t s, const DeltaShape &d, const float *qkv, const float *beta, const float *lg, float *state, int M, int pos0, float *rec,
                        int64_t rec_floats, float *o, const float *gate, const float *normw, void *outa, int64_t lda, int prec) {
    if (d.D > 256 || d.V > 256 || M < 1) return hipErrorInvalidValue;
    if (!delta_wide_chunks(d, M)) {
        if (rec_floats < delta_rec16_floats(d, M)) return hipErrorInvalidValue;
        const auto launch = d.D > 192 ? delta_walk16_launch<4> : d.D > 128 ? delta_walk16_launch<3> : d.D > 64 ? delta_walk16_launch<2> : delta_walk16_launch<1>;
        const hipError_t e = launch(s, d, qkv, beta, lg, state, M, pos0, rec, o);
        return e != hipSuccess ? e : k_head_norm_rows(s, o, gate, normw, M, d.H, d.V, d.eps, outa, lda, prec);
    }
    // passes over as many chunks as have their records in memory together; a pass goes on from the state as the positions of a later call do
    const int n = WK_T * delta_pass_chunks(d, M, rec_floats);
    if (n < 1) return hipErrorInvalidValue;
    const auto launch = d.D > 192 ? delta_walk_launch<4> : d.D > 128 ? delta_walk_launch<3> : d.D > 64 ? delta_walk_launch<2> : delta_walk_launch<1>;
    for (int64_t m = 0; m < M; m += n) {
        const hipError_t e = launch(s, d, qkv + m * d.channels(), beta + m * d.H, lg + m * d.H * d.D, state, std::min(n, M - (int)m), pos0 + (int)m, rec,
                                    gate + m * d.H * d.V, normw, prec ? (void *)((float *)outa + m * lda) : (void *)((uint16_t *)outa + m * lda), lda, prec);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// one wavefront per (token, head)
template <int PREC>
__global__ __launch_bounds__(256) void head_norm_rows_kernel(const float *o, const float *gate, const float *normw, int M, int H, int V,
                                                             float eps, void *outa, int64_t lda) {
    const int lane = threadIdx.x & 63;
    const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (unit >= (int64_t)M * H) return;
    const int m = (int)(unit / H), h = (int)(unit - (int64_t)m * H);
    const float *x = o + (int64_t)m * H * V + h * V, *g = gate + (int64_t)m * H * V + h * V;
    float ss = 0.0f;
    for (int j = lane; j < V; j += 64) ss = fmaf(x[j], x[j], ss);
    const float r = 1.0f / sqrtf(l_wave_sum(ss) / (float)V + eps);
    for (int j = lane; j < V; j += 64) l_store_act<PREC>(outa, m * lda + h * V + j, x[j] * r * normw[j] * g[j]);
    if (h == H - 1)
        for (int64_t j = (int64_t)H * V + lane; j < lda; j += 64) l_store_act<PREC>(outa, m * lda + j, 0.0f);
}
hipError_t k_head_norm_rows(hipStream_t s, const float *o, const float *gate, const float *normw, int M, int H, int V, float eps,
                            void *outa, int64_t lda, int prec) {
    const dim3 grid((unsigned)(((int64_t)M * H + 3) / 4));
    if (prec)
        hipLaunchKernelGGL((head_norm_rows_kernel<1>), grid, dim3(256), 0, s, o, gate, normw, M, H, V, eps, outa, lda);
    else
        hipLaunchKernelGGL((head_norm_rows_kernel<0>), grid, dim3(256), 0, s, o, gate, normw, M, H, V, eps, outa, lda);
    return hipGetLastError();
}
