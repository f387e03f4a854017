// Small per-token kernels: weight repack, embedding lookup, rmsnorm + q8_K quantize,
// SwiGLU + quantize, RoPE + KV append, argmax, layout helpers.
#include <hip/hip_fp16.h>
#include <mutex>

#include "dev_common.h"
#include "draw.h"

// ------------------------------------------------------------------------------------------
// Repack GGUF super-blocks <-> field streams (see DevTensor).  One thread per 16-bit word
// of the raw block keeps it valid for q6_K, whose 210-byte blocks are only 2-byte aligned.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ int64_t stream_word_index(int type, int64_t blk, int w, int &which) {
    // returns the index (in 16-bit words) inside stream `which` for word w of block blk
    // which: 0 hdr, 1 qs/ql, 2 qh, 3 sc6, 4 d6
    if (type == L2H_TYPE_Q4_K) {
        if (w < 8) { which = 0; return blk * 8 + w; }
        which = 1; return blk * 64 + (w - 8);
    }
    if (type == L2H_TYPE_Q5_K) {
        if (w < 8) { which = 0; return blk * 8 + w; }
        if (w < 24) { which = 2; return blk * 16 + (w - 8); }
        which = 1; return blk * 64 + (w - 24);
    }
    // Q6_K: ql 64 words, qh 32 words, scales 8 words (bytes permuted, handled by caller), d 1 word
    if (w < 64) { which = 1; return blk * 64 + w; }
    if (w < 96) { which = 2; return blk * 32 + (w - 64); }
    if (w < 104) { which = 3; return blk * 8 + (w - 96); }
    which = 4; return blk;
}

__global__ __launch_bounds__(256) void repack_kernel(DevTensor t, const uint16_t *raw, uint16_t *raw_out,
                                                     int64_t nblocks, int words_per_block, bool inverse) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= nblocks * words_per_block) return;
    const int64_t blk = gid / words_per_block;
    const int w = (int)(gid % words_per_block);
    int which;
    const int64_t idx = stream_word_index(t.type, blk, w, which);
    uint16_t *streams[5] = {(uint16_t *)t.hdr, (uint16_t *)t.qs, (uint16_t *)t.qh, (uint16_t *)t.sc6,
                            (uint16_t *)t.d6};
    if (which == 3) {
        // q6_K scales: original byte o = 8n + hh + 2g  <->  stream byte p = 4*(2n+hh) + g
        uint8_t *sc = (uint8_t *)t.sc6 + blk * 16;
        const uint8_t *rb = (const uint8_t *)raw + blk * 210 + 192;
        uint8_t *ro = (uint8_t *)raw_out + blk * 210 + 192;
        for (int k = 0; k < 2; k++) {
            const int o = 2 * (w - 96) + k;
            const int n = o >> 3, hh = o & 1, g = (o & 7) >> 1;
            const int p = 4 * (2 * n + hh) + g;
            if (inverse)
                ro[o] = sc[p];
            else
                sc[p] = rb[o];
        }
        return;
    }
    if (inverse)
        raw_out[gid] = streams[which][idx];
    else
        streams[which][idx] = raw[gid];
}

hipError_t k_repack(hipStream_t s, const DevTensor &t, const void *raw_dev, bool inverse, void *raw_out) {
    const int wpb = (int)(l2h_gguf_block_bytes(t.type) / 2);
    const int64_t nblocks = t.ne1 * t.nb;
    const int64_t total = nblocks * wpb;
    const int64_t grid = (total + 255) / 256;
    hipLaunchKernelGGL(repack_kernel, dim3((unsigned)grid), dim3(256), 0, s, t, (const uint16_t *)raw_dev,
                       (uint16_t *)raw_out, nblocks, wpb, inverse);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// dequantize!(x, token_embedding_table[:, token])  (reference src/inference.jl:236)
// The token of the step is prompt[step] while inside the prompt, else the previous argmax
// (src/inference.jl:354-360,385).
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void embed_kernel(DevTensor emb, const DecodeCtl *ctl, const int32_t *prompt,
                                                    float *x, float *rope_cs, int hs, float theta_scale) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < (hs >> 1)) {
        // cos/sin of this position's RoPE angles, shared by all layers and heads: theta_i is
        // fp32(pos) advanced by i fp32 multiplications (reference src/inference.jl:122-127)
        float theta = 1.0f * (float)ctl->pos;
        for (int k = 0; k < (int)threadIdx.x; k++) theta *= theta_scale;
        rope_cs[2 * threadIdx.x] = (float)cos((double)theta);
        rope_cs[2 * threadIdx.x + 1] = (float)sin((double)theta);
    }
    if (i >= emb.ne0) return;
    const int tok = ctl->step < ctl->n_prompt ? prompt[ctl->step] : ctl->last_argmax;
    x[i] = dequant_elem(emb, tok, i);
}

hipError_t k_embed(hipStream_t s, const DevTensor &emb, const DecodeCtl *ctl, const int32_t *prompt, float *x,
                   float *rope_cs, int head_size, float theta_scale) {
    hipLaunchKernelGGL(embed_kernel, dim3((unsigned)((emb.ne0 + 255) / 256)), dim3(256), 0, s, emb, ctl, prompt, x,
                       rope_cs, head_size, theta_scale);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void dequant_kernel(DevTensor t, int64_t row0, int64_t nrows, float *y) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= nrows * t.ne0) return;
    y[gid] = dequant_elem(t, row0 + gid / t.ne0, gid % t.ne0);
}

hipError_t k_dequant(hipStream_t s, const DevTensor &t, int64_t row0, int64_t nrows, float *y) {
    const int64_t total = nrows * t.ne0;
    hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, t, row0, nrows, y);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// hb[i] = hb[i] * (1/(1+exp(-hb[i]))) * hb2[i]  (reference src/inference.jl:295-299),
// exp evaluated in fp64 and rounded to fp32.  Stand-alone form, used when w1 and w3 differ in
// type and cannot share one launch.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void swiglu_kernel(float *hb, const float *hb2, int n) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const float a = hb[t];
    const float e = (float)exp((double)(-a));
    const float v = a * (1.0f / (1.0f + e));
    hb[t] = v * hb2[t];
}

hipError_t k_swiglu(hipStream_t s, float *hb, const float *hb2, int n) {
    hipLaunchKernelGGL(swiglu_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, hb, hb2, n);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// rope!(x) (reference src/inference.jl:112-167), stand-alone form.
// theta of pair i is fp32(pos) advanced by i fp32 multiplications with theta_scale
// (:122-127); cos/sin are evaluated in fp64 and rounded to fp32; the complex product
// rounds each of its four products (Complex{Float32} multiplication).
// K cache layout per layer: [n_kv_heads][hs/4][seq_len][4]; V cache: [n_kv_heads][seq_len][hs].
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ void rope_pair(float a, float b, int i, int pos, float theta_scale, float &re, float &im) {
    float theta = 1.0f * (float)pos;
    for (int k = 0; k < i; k++) theta *= theta_scale;
    const float c = (float)cos((double)theta);
    const float s = (float)sin((double)theta);
    const float ac = a * c, bs = b * s, as = a * s, bc = b * c;
    re = ac - bs;
    im = as + bc;
}

__device__ __forceinline__ int64_t kc_index(int kvh, int i, int t, int hs, int seq_len) {
    return (((int64_t)kvh * (hs >> 2) + (i >> 2)) * seq_len + t) * 4 + (i & 3);
}

__global__ __launch_bounds__(256) void rope_only_kernel(float *x, int hs, int n_heads, int pos, float theta_scale,
                                                        int neox) {
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int half = hs >> 1;
    if (gid >= n_heads * half) return;
    const int h = gid / half, i = gid % half;
    const int e0 = neox ? i : 2 * i, e1 = neox ? half + i : 2 * i + 1;
    float re, im;
    rope_pair(x[h * hs + e0], x[h * hs + e1], i, pos, theta_scale, re, im);
    x[h * hs + e0] = re;
    x[h * hs + e1] = im;
}

hipError_t k_rope_only(hipStream_t s, float *x, int head_size, int n_heads, int pos, float theta_scale, int neox) {
    const int total = n_heads * head_size / 2;
    hipLaunchKernelGGL(rope_only_kernel, dim3((total + 255) / 256), dim3(256), 0, s, x, head_size, n_heads, pos,
                       theta_scale, neox);
    return hipGetLastError();
}

// canonical [n][kv_dim] rows <-> cache layouts, positions pos0 .. pos0+n-1 of one layer
__global__ __launch_bounds__(256) void kv_layout_kernel(float *kc, float *vc, float *k_lin, float *v_lin, int pos0,
                                                        int n, int hs, int n_kv_heads, int seq_len, int to_cache, int kv16) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int kv_dim = hs * n_kv_heads;
    if (gid >= (int64_t)n * kv_dim) return;
    const int r = (int)(gid / kv_dim), e = (int)(gid % kv_dim);
    const int h = e / hs, i = e % hs, t = pos0 + r;
    const int64_t ki = kc_index(h, i, t, hs, seq_len);
    const int64_t vi = ((int64_t)h * seq_len + t) * hs + i;
    if (kv16) {  // fp16 cache: rounded to nearest even on the way in, widened exactly on the way out
        __half *kh = (__half *)kc, *vh = (__half *)vc;
        const int64_t ki = kc16_index(h, i, t, hs, seq_len);  // (the fp16 K cache groups eight elements)
        if (to_cache) {
            kh[ki] = __float2half_rn(k_lin[gid]);
            vh[vi] = __float2half_rn(v_lin[gid]);
        } else {
            k_lin[gid] = __half2float(kh[ki]);
            v_lin[gid] = __half2float(vh[vi]);
        }
        return;
    }
    if (to_cache) {
        kc[ki] = k_lin[gid];
        vc[vi] = v_lin[gid];
    } else {
        k_lin[gid] = kc[ki];
        v_lin[gid] = vc[vi];
    }
}

hipError_t k_kv_layout(hipStream_t s, float *kc, float *vc, float *k_lin, float *v_lin, int pos0, int n, int head_size,
                       int n_kv_heads, int seq_len, bool to_cache, int kv16) {
    const int64_t total = (int64_t)n * head_size * n_kv_heads;
    hipLaunchKernelGGL(kv_layout_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, kc, vc, k_lin, v_lin,
                       pos0, n, head_size, n_kv_heads, seq_len, to_cache ? 1 : 0, kv16);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// argmax(logits): first maximal index (reference src/inference.jl:360).  Stage 2 also advances the control
// block to the next step.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ unsigned long long block_max_u64(unsigned long long key, unsigned long long *red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    key = wave_max_u64(key);
    __syncthreads();
    if (lane == 0) red[wave] = key;
    __syncthreads();
    unsigned long long t = red[0];
    for (int w = 1; w < nw; w++) t = red[w] > t ? red[w] : t;
    return t;
}

__global__ __launch_bounds__(256) void argmax_stage1_kernel(const float *x, int64_t n, unsigned long long *partial) {
    __shared__ unsigned long long red[4];
    unsigned long long best = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const unsigned long long key = argmax_key(x[i], (uint32_t)i);
        best = key > best ? key : best;
    }
    best = block_max_u64(best, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = best;
}

// the control block goes on to the next step, whose token is the largest key's
__device__ __forceinline__ int argmax_index(unsigned long long key) { return (int)(0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFull)); }
__device__ __forceinline__ void argmax_advance(unsigned long long best, DecodeCtl *ctl, int32_t *out_tokens, int max_out) {
    const int idx = argmax_index(best);
    ctl->last_argmax = idx;
    if (ctl->step >= ctl->n_prompt - 1 && ctl->n_out < max_out) {
        out_tokens[ctl->n_out] = idx;
        ctl->n_out += 1;
    }
    ctl->step += 1;
    ctl->pos += 1;
}

__global__ __launch_bounds__(256) void argmax_stage2_kernel(const unsigned long long *partial, int nparts,
                                                            DecodeCtl *ctl, int32_t *out_tokens, int max_out) {
    __shared__ unsigned long long red[4];
    unsigned long long best = 0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) best = partial[i] > best ? partial[i] : best;
    best = block_max_u64(best, red);
    if (threadIdx.x == 0) argmax_advance(best, ctl, out_tokens, max_out);
}

// Both stages by one workgroup, all of a thread's elements under way at once: 32 000 logits in 5.8 us, against 4.6 + 4.1 in two
// launches.  Bound by what one CU draws from the L2s; beyond 32 768 elements a thread's would no longer fit its registers.
// At the end of a prompt pass, launch by launch: 4 us less (1244 -> 1239 us, 33 positions of 4096 wide layers).  In a recorded step, whose launches
// follow each other closely and whose next one waits for this, 0.8 to 1.4 us more (a token of Vudelix, width 768, 4 layers: 170.6 us with two launches,
// 171.7 with one; 2176, 2 layers: 140.5, 141.7): steps take two.
#define ARGMAX_ONE_N 32768
__global__ __launch_bounds__(1024) void argmax_one_kernel(const float *x, int n, DecodeCtl *ctl, int32_t *out_tokens, int max_out) {
    __shared__ unsigned long long red[16];
    constexpr int Q = ARGMAX_ONE_N / 4096;
    const int t = threadIdx.x;
    float4 v[Q];
#pragma unroll
    for (int u = 0; u < Q; u++) v[u] = *(const float4 *)(x + max(0, min(4 * (t + 1024 * u), (n & ~3) - 4)));
    const int tail = (n & ~3) + t;
    unsigned long long best = tail < n ? argmax_key(x[tail], (uint32_t)tail) : 0ull;
#pragma unroll
    for (int u = 0; u < Q; u++) {
        const int i = 4 * (t + 1024 * u);
        if (i + 3 < n) {
            const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned long long key = argmax_key(e[k], (uint32_t)(i + k));
                best = key > best ? key : best;
            }
        }
    }
    best = block_max_u64(best, red);
    if (t == 0) argmax_advance(best, ctl, out_tokens, max_out);
}

hipError_t k_argmax(hipStream_t s, const float *x, int64_t n, int64_t *partial, DecodeCtl *ctl, int32_t *out_tokens,
                    int max_out, bool step) {
    if (!step && n >= 4 && n <= ARGMAX_ONE_N && (uintptr_t)x % 16 == 0) {
        hipLaunchKernelGGL(argmax_one_kernel, dim3(1), dim3(1024), 0, s, x, (int)n, ctl, out_tokens, max_out);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(argmax_stage1_kernel, dim3(L2H_ARGMAX_BLOCKS), dim3(256), 0, s, x, n,
                       (unsigned long long *)partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(argmax_stage2_kernel, dim3(1), dim3(256), 0, s, (const unsigned long long *)partial,
                       L2H_ARGMAX_BLOCKS, ctl, out_tokens, max_out);
    return hipGetLastError();
}

// The largest of the keys that a layered model's last step has left (k_rows_keys): the control block goes on.  Behind the last step of a call; between
// two steps step_begin_kernel does it.
hipError_t k_argmax_keys(hipStream_t s, const unsigned long long *keys, int n, DecodeCtl *ctl, int32_t *out_tokens, int max_out) {
    hipLaunchKernelGGL(argmax_stage2_kernel, dim3(1), dim3(256), 0, s, keys, n, ctl, out_tokens, max_out);
    return hipGetLastError();
}

// The beginning of a layered model's step: the token that the step before has left the keys of, then embed_kernel's work.  Every workgroup picks for
// itself, from the copy of the control block that the step before made (`prev`; a call's first step finds the caller's, without keys); the
// first one advances the control block.  One launch where there were three (embedding, two for the argmax): 32 tokens of Lezepel, width 2048, 4 layers
// 8.96 -> 8.85 ms with the keys' 1 us in the classifier.
// Workgroups from n_x on copy the token's row of the per-token table, of which every layer's side input reads a part (with the token and then the
// element two loads away from each of those launches: 3.7 us for 256 rows of 768, 2.9 like this).
__global__ __launch_bounds__(256) void step_begin_kernel(DevTensor emb, const DecodeCtl *prev, DecodeCtl *ctl, const unsigned long long *keys, int n_keys,
                                                         const int32_t *prompt, int32_t *out_tokens, int max_out, float *x, float scale, float *x_copy,
                                                         StepSide side, int n_x) {
    __shared__ unsigned long long red[4];
    DecodeCtl c = *prev;
    unsigned long long best = 0;
    for (int i = threadIdx.x; i < n_keys; i += 256) best = keys[i] > best ? keys[i] : best;
    if (c.picks) {
        best = block_max_u64(best, red);
        const int idx = argmax_index(best);
        c.last_argmax = idx;
        if (c.step >= c.n_prompt - 1 && c.n_out < max_out) {
            if (blockIdx.x == 0 && threadIdx.x == 0) out_tokens[c.n_out] = idx;
            c.n_out += 1;
        }
        c.step += 1;
        c.pos += 1;
        c.picks = 0;
        if (blockIdx.x == 0 && threadIdx.x == 0) *ctl = c;
    }
    const int tok = c.step < c.n_prompt ? prompt[c.step] : c.last_argmax;
    if ((int)blockIdx.x >= n_x) {
        const int64_t i = (int64_t)((int)blockIdx.x - n_x) * 256 + threadIdx.x;
        if (i < side.n) side.row[i] = side.table[tok * side.n + i];
        return;
    }
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= emb.ne0) return;
    const float v = scale * dequant_elem(emb, tok, i);
    x[i] = v;
    if (x_copy) x_copy[i] = v;
}
hipError_t k_step_begin(hipStream_t s, const DevTensor &emb, const DecodeCtl *prev, DecodeCtl *ctl, const unsigned long long *keys, int n_keys,
                        const int32_t *prompt, int32_t *out_tokens, int max_out, float *x, float scale, float *x_copy, const StepSide &side) {
    const int64_t n_x = (emb.ne0 + 255) / 256, n_side = (side.n + 255) / 256;
    hipLaunchKernelGGL(step_begin_kernel, dim3((unsigned)(n_x + n_side)), dim3(256), 0, s, emb, prev, ctl, keys, n_keys, prompt, out_tokens, max_out,
                       x, scale, x_copy, side, (int)n_x);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// argmax for callers that cannot allocate (code under stream capture, serving loops, harnesses that forbid
// hipMalloc): the same two stages, with the per-workgroup keys of stage 1 in a file-scope device array
// instead of an allocation.  Every GPU the library runs on holds its own copy of the array (2 KiB) until
// the process ends; calls that overlap on one GPU would share it and race.
// ------------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned long long scratch[L2H_ARGMAX_BLOCKS];

// In host code `scratch` is a stand-in, not a device address: each device's address is asked for once, with
// that device current, and kept.
#define L2H_MAX_DEVICES 64
static unsigned long long *g_scratch_ptr[L2H_MAX_DEVICES];

static std::mutex g_scratch_mu;

hipError_t k_noalloc_init(int device) {
    if (device < 0 || device >= L2H_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return hipSuccess;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[device] = (unsigned long long *)p;
    return hipSuccess;
}

__global__ __launch_bounds__(256) void argmax_stage2_plain_kernel(const unsigned long long *partial, int nparts,
                                                                  int32_t *out) {
    __shared__ unsigned long long red[4];
    unsigned long long best = 0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) best = partial[i] > best ? partial[i] : best;
    best = block_max_u64(best, red);
    if (threadIdx.x == 0) *out = (int32_t)(0xFFFFFFFFu - (uint32_t)(best & 0xFFFFFFFFull));
}

// x and out are device pointers; nothing is allocated, nothing is waited for.  Stage 1 writes every one of
// the L2H_ARGMAX_BLOCKS keys on every call (a workgroup without elements writes the smallest key), so what
// the previous call left in the array is never read.
hipError_t k_argmax_noalloc(hipStream_t s, int device, const float *x, int64_t n, int32_t *out) {
    if (device < 0 || device >= L2H_MAX_DEVICES || !g_scratch_ptr[device]) return hipErrorNotInitialized;
    unsigned long long *partial = g_scratch_ptr[device];
    hipLaunchKernelGGL(argmax_stage1_kernel, dim3(L2H_ARGMAX_BLOCKS), dim3(256), 0, s, x, n, partial);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(argmax_stage2_plain_kernel, dim3(1), dim3(256), 0, s, (const unsigned long long *)partial,
                       L2H_ARGMAX_BLOCKS, out);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// softmax!(x) (reference src/inference.jl:169-174), single vector, one workgroup.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void softmax_kernel(float *x, int64_t n) {
    __shared__ double redd[16];
    __shared__ float redf[16];
    float mx = -INFINITY;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) mx = fmaxf(mx, x[i]);
    mx = block_max_f32(mx, redf);
    double acc = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const float e = (float)exp((double)(x[i] - mx));
        x[i] = e;
        acc += (double)e;
    }
    const float sf = (float)block_sum_f64(acc, redd);
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) x[i] = x[i] / sf;
}

hipError_t k_softmax(hipStream_t s, float *x, int64_t n) {
    hipLaunchKernelGGL(softmax_kernel, dim3(1), dim3(256), 0, s, x, n);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// plain streaming read (measured HBM ceiling) and fp32 -> fp64 widening
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void stream_read_kernel(const uint4 *p, int64_t n16, uint32_t *sink) {
    uint32_t acc = 0;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n16; i += 4 * stride) {
        const uint4 a = p[i], b = p[i + stride], c = p[i + 2 * stride], d = p[i + 3 * stride];
        acc ^= a.x ^ a.y ^ a.z ^ a.w ^ b.x ^ b.y ^ b.z ^ b.w ^ c.x ^ c.y ^ c.z ^ c.w ^ d.x ^ d.y ^ d.z ^ d.w;
    }
    for (; i < n16; i += stride) {
        const uint4 a = p[i];
        acc ^= a.x ^ a.y ^ a.z ^ a.w;
    }
    if (acc == 0x9E3779B9u) sink[0] = acc;  // practically never true: keeps the loads alive
}

hipError_t k_stream_read(hipStream_t s, const uint4 *p, int64_t n16, uint32_t *sink) {
    hipLaunchKernelGGL(stream_read_kernel, dim3(256 * 8), dim3(256), 0, s, p, n16, sink);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void f32_to_f64_kernel(const float *x, double *y, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = (double)x[i];
}

hipError_t k_f32_to_f64(hipStream_t s, const float *x, double *y, int64_t n) {
    hipLaunchKernelGGL(f32_to_f64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, y, n);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// temperature sampling (reference src/inference.jl:363-367): logits ./= T; softmax!; wsample.
// wsample's walk is reproduced with a host-supplied uniform number u in [0, 1): the pick is the first
// index whose cumulative weight reaches u * sum(weights).  exp in fp64 rounded to fp32 and the sums
// in fp64 (as everywhere in this library).
// ------------------------------------------------------------------------------------------
// In three launches over SAMPLE_PARTS workgroups at most, each a run of the logits, because a run's exponentials need the largest of all and its probabilities the
// sum of all; the workgroup that is through last picks, so that nobody waits.  (One workgroup alone: 558 us for 128 256 of them, 125 exponentials in fp64 a
// thread; a fourth launch for the pick: 5 us more.)  Up to SAMPLE_ONE logits one workgroup does it all, whose elements stay in registers.
// part: the runs' largest values, sums of exponentials, sums of probabilities.
#define SAMPLE_THREADS 256
#define SAMPLE_PARTS 256
struct SampleRun {
    int lo, hi;
};
__device__ __forceinline__ SampleRun sample_run(int n, int per, int b) {
    return SampleRun{(int)min((int64_t)n, (int64_t)b * per), (int)min((int64_t)n, (int64_t)(b + 1) * per)};
}
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_max_kernel(const float *logits, int n, int per, float temperature, float *p, double *part) {
    __shared__ float red[SAMPLE_THREADS / 64];
    const SampleRun r = sample_run(n, per, blockIdx.x);
    float mx = -INFINITY;
    for (int i = r.lo + threadIdx.x; i < r.hi; i += SAMPLE_THREADS) {
        const float v = logits[i] / temperature;
        p[i] = v;
        mx = fmaxf(mx, v);
    }
    mx = block_max_f32(mx, red);
    if (threadIdx.x == 0) part[blockIdx.x] = (double)mx;
}
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_exp_kernel(int n, int per, int parts, float *p, double *part) {
    __shared__ float redf[SAMPLE_THREADS / 64];
    __shared__ double red[SAMPLE_THREADS / 64];
    const SampleRun r = sample_run(n, per, blockIdx.x);
    const float mx = block_max_f32((int)threadIdx.x < parts ? (float)part[threadIdx.x] : -INFINITY, redf);
    double sum = 0.0;
    for (int i = r.lo + threadIdx.x; i < r.hi; i += SAMPLE_THREADS) {
        const float e = (float)exp((double)(p[i] - mx));
        p[i] = e;
        sum += (double)e;
    }
    sum = block_sum_f64(sum, red);
    if (threadIdx.x == 0) part[SAMPLE_PARTS + blockIdx.x] = sum;
}
// Running sums over the workgroup's values: in front of this thread's and behind it (draw.h: a thread's end is the next one's lower, bit for bit); all: behind
// the last.  red: a double a wavefront
struct SampleEnds {
    double lower, end, all;
};
__device__ __forceinline__ SampleEnds sample_ends(double v, double *red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    double x = v;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const double o = __shfl_up(x, d, WAVE);
        x += lane >= d ? o : 0.0;
    }
    const double up = __shfl_up(x, 1, WAVE);
    __syncthreads();
    if (lane == 63) red[wave] = x;
    __syncthreads();
    double base = 0.0, all = 0.0;
    for (int w = 0; w < nw; w++) {
        if (w == wave) base = all;
        all += red[w];
    }
    return {base + (lane ? up : 0.0), base + x, all};
}
// the thread that takes a draw of such sums; s_own: two words of LDS that nobody else uses
__device__ __forceinline__ void sample_owner_clear(int *s_own) {  // (by one thread, a barrier before sample_owner)
    s_own[0] = 0x7FFFFFFF;
    s_own[1] = -1;
}
__device__ __forceinline__ int sample_owner(double own, double end, double target, int *s_own) {
    const int wave0 = threadIdx.x & ~63;
    const unsigned long long weight = __ballot(own > 0.0), reach = __ballot(draw_reaches(own, end, target));
    if ((threadIdx.x & 63) == 0 && reach) atomicMin(s_own, wave0 + __ffsll(reach) - 1);
    if ((threadIdx.x & 63) == 0 && weight) atomicMax(s_own + 1, wave0 + 63 - __clzll((long long)weight));
    __syncthreads();
    return s_own[0] == 0x7FFFFFFF ? s_own[1] : s_own[0];
}
__device__ __forceinline__ float sample_load(const float *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// Probabilities and their sums; then, by the workgroup that is through last (count: zero between launches), the pick: the run that the target, u times the
// whole, lies in, then the element.
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_prob_kernel(int n, int per, int parts, float u, float *p, double *part, unsigned *count, int32_t *out) {
    __shared__ double red[SAMPLE_THREADS / 64], s_lower;
    __shared__ int s_last, s_run[2], s_own[2];
    const int t = threadIdx.x;
    {
        const SampleRun r = sample_run(n, per, blockIdx.x);
        const float sf = (float)block_sum_f64(t < parts ? part[SAMPLE_PARTS + t] : 0.0, red);
        double sum = 0.0;
        for (int i = r.lo + t; i < r.hi; i += SAMPLE_THREADS) {
            const float pr = p[i] / sf;
            __hip_atomic_store(p + i, pr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // (read by another workgroup)
            sum += (double)pr;
        }
        __syncthreads();
        sum = block_sum_f64(sum, red);
        if (t == 0) __hip_atomic_store(part + 2 * SAMPLE_PARTS + blockIdx.x, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (they are in memory before the count says so)
    __syncthreads();
    if (t == 0) {
        s_last = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)parts - 1u;
        if (s_last) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sample_owner_clear(s_run);
        sample_owner_clear(s_own);
    }
    __syncthreads();
    if (!s_last) return;
    const double v = t < parts ? __hip_atomic_load(part + 2 * SAMPLE_PARTS + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
    const SampleEnds runs = sample_ends(v, red);
    const double target = (double)u * runs.all;
    if (!(runs.all > 0.0)) {  // (the probabilities are not numbers: one of the logits was none, or was not finite once divided)
        if (t == 0) *out = -1;
        return;
    }
    const int at = sample_owner(v, runs.end, target, s_run);
    if (t == at) s_lower = runs.lower;
    const SampleRun r = sample_run(n, per, at);
    const int each = (per + SAMPLE_THREADS - 1) / SAMPLE_THREADS, lo = min(r.hi, r.lo + t * each), hi = min(r.hi, lo + each);
    double mine = 0.0;
    for (int i = lo; i < hi; i++) mine += (double)sample_load(p + i);
    const SampleEnds own = sample_ends(mine, red);  // (s_lower is behind its barriers)
    if (t != sample_owner(mine, s_lower + own.end, target, s_own)) return;
    DrawWalk walk(s_lower + own.lower, target);
    for (int i = lo; i < hi; i++) walk.next(i, sample_load(p + i));
    *out = target > 0.0 ? walk.pick : 0;  // (u = 0 is reached by the first of all)
}

// the same for up to SAMPLE_ONE logits, four a thread
#define SAMPLE_ONE 4096
__global__ __launch_bounds__(1024) void sample_one_kernel(const float *logits, int n, float temperature, float u, float *p, int32_t *out) {
    __shared__ float redf[16];
    __shared__ double red[16];
    __shared__ int s_own[2];
    const int t = threadIdx.x, i0 = 4 * t;
    float v[4], mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] = i0 + k < n ? logits[i0 + k] / temperature : -INFINITY;
        mx = fmaxf(mx, v[k]);
    }
    mx = block_max_f32(mx, redf);
    double sum = 0.0;
#pragma nounroll
    for (int k = 0; k < 4; k++) {  // (one exponential's code)
        const float x = k == 0 ? v[0] : k == 1 ? v[1] : k == 2 ? v[2] : v[3];
        const float e = i0 + k < n ? (float)exp((double)(x - mx)) : 0.0f;
        if (k == 0) v[0] = e;
        if (k == 1) v[1] = e;
        if (k == 2) v[2] = e;
        if (k == 3) v[3] = e;
        sum += (double)e;
    }
    const float sf = (float)block_sum_f64(sum, red);
    double own = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        v[k] /= sf;
        if (i0 + k >= n) break;
        p[i0 + k] = v[k];
        own += (double)v[k];
    }
    if (t == 0) sample_owner_clear(s_own);
    const SampleEnds ends = sample_ends(own, red);
    const double target = (double)u * ends.all;
    if (!(ends.all > 0.0)) {  // (not numbers)
        if (t == 0) *out = -1;
        return;
    }
    if (t != sample_owner(own, ends.end, target, s_own)) return;
    DrawWalk walk(ends.lower, target);
#pragma unroll
    for (int k = 0; k < 4; k++)
        if (i0 + k < n) walk.next(i0 + k, v[k]);
    *out = target > 0.0 ? walk.pick : 0;
}

hipError_t k_sample(hipStream_t s, const float *logits, int n, float temperature, float u, float *p, double *part, unsigned *count, int32_t *out) {
    if (n <= SAMPLE_ONE) {
        hipLaunchKernelGGL(sample_one_kernel, dim3(1), dim3(1024), 0, s, logits, n, temperature, u, p, out);
        return hipGetLastError();
    }
    const int per = std::max(1024, (int)(((int64_t)n + SAMPLE_PARTS - 1) / SAMPLE_PARTS)), parts = (int)(((int64_t)n + per - 1) / per);
    hipLaunchKernelGGL(sample_max_kernel, dim3(parts), dim3(SAMPLE_THREADS), 0, s, logits, n, per, temperature, p, part);
    hipLaunchKernelGGL(sample_exp_kernel, dim3(parts), dim3(SAMPLE_THREADS), 0, s, n, per, parts, p, part);
    hipLaunchKernelGGL(sample_prob_kernel, dim3(parts), dim3(SAMPLE_THREADS), 0, s, n, per, parts, u, p, part, count, out);
    return hipGetLastError();
}

// Up to WORD_COPIES runs of 4-byte words from and to anywhere the device sees: what a call hands over and gets back, in one launch of 2 us where a copy of each is one of
// 4 to 5 and twice the work for the host.
__global__ __launch_bounds__(1024) void words_kernel(WordCopies c) {
    const WordCopy w = c.run[blockIdx.x];
    for (int64_t i = threadIdx.x; i < w.n; i += 1024) w.to[i] = w.from[i];
}
hipError_t k_words(hipStream_t s, const WordCopies &c) {
    int n = 0;
    WordCopies d;
    for (const WordCopy &w : c.run)
        if (w.n > 0) d.run[n++] = w;
    if (!n) return hipSuccess;
    hipLaunchKernelGGL(words_kernel, dim3((unsigned)n), dim3(1024), 0, s, d);
    return hipGetLastError();
}
