// The product loop of the kernels for few positions (bf16, matrices read once): 32 or 64 rows of a matrix x 32 or 64 positions a workgroup, by four wavefronts
// that do not wait for each other.
//
// What bounds such a product is what a compute unit can have under way: so each wavefront takes every fourth step of 64 inputs and brings its rows' and
// positions' 128-byte lines straight into a ring of its own in LDS (16 bytes a lane), two to four steps ahead of the matrix instructions, 128 to 144 KB a
// compute unit.  Only the order of its own loads tells when a step has landed, so the loop has no barrier; the four sums are added at the end, in order.
#pragma once

#include "pf_tile.h"

constexpr int few_ring_block(int tn, int tm) { return 128 * (tn + tm); }                   // bytes of a step: rows, then positions
constexpr int few_ring_depth(int tn, int tm) { return 147456 / (4 * few_ring_block(tn, tm)); }  // steps of a wavefront
constexpr int few_ring_lds(int tn, int tm) { return 4 * few_ring_depth(tn, tm) * few_ring_block(tn, tm); }
constexpr int FEW_RING_SUMS = 8 * 33;  // 16-byte words of 32 rows x 32 positions: row quad q of position p at 33 q + p
// which row, and which 16 bytes of its 64 inputs, load i of a lane brings: chunk c of row r lies in place c ^ pf_swz(r)
__device__ __forceinline__ int few_ring_row(int i, int lane) { return 8 * i + (lane >> 3); }
__device__ __forceinline__ int few_ring_chunk(int i, int lane) { return (lane & 7) ^ pf_swz(few_ring_row(i, lane)); }

// Which steps a wavefront takes, and in which order: every fourth one, from `first` on among its own (modulo their number): rows lie a multiple of 4 KB apart, so
// workgroups in step would all ask the same channels.  (16 384 rows x 2048 inputs, 8 to 32 positions: 19.4 us without, 15.9 with it.)
struct FewQuarters {
    int n, from, wave;
    __device__ __forceinline__ FewQuarters(int nk, unsigned first, int wave) : n(nk > wave ? (nk - wave + 3) >> 2 : 0), from(0), wave(wave) {
        if (n) from = (int)(first % (unsigned)n);
    }
    __device__ __forceinline__ int step(int i) const {
        const int j = i + from;
        return wave + 4 * (j < n ? j : j - n);
    }
    __device__ __forceinline__ int cut() const { return -1; }
};
// Or two eighths of the inputs, w and w + 4, each summed by itself in order: the same sums whichever comes first.
struct FewEighths {
    int n, at[2], before;
    __device__ __forceinline__ FewEighths(int nk, unsigned first, int wave) {
        const int lo = nk * wave / 8, n_lo = nk * (wave + 1) / 8 - lo, hi = nk * (wave + 4) / 8, n_hi = nk * (wave + 5) / 8 - hi;
        const bool turned = first & 1u;
        before = turned ? n_hi : n_lo;
        at[0] = turned ? hi : lo;
        at[1] = (turned ? lo : hi) - before;
        n = n_lo + n_hi;
    }
    __device__ __forceinline__ int step(int i) const { return i + at[i >= before]; }
    __device__ __forceinline__ int cut() const { return before; }
};

// a(i, k): address of the 16 bytes that load i of this lane brings of the rows' step k; x(i, k): of the positions'.  nk: steps.  s: few_ring_lds() bytes.  Behind the call s holds wavefront w's sums in words
// [w][rows / 32][positions / 32][FEW_RING_SUMS], and all wavefronts have met.
template <int TN, int TM, class Order, class A, class X>
__device__ __forceinline__ void few_ring(int nk, unsigned first, unsigned char *s, A a, X x) {
    constexpr int BLOCK = few_ring_block(TN, TM), DEPTH = few_ring_depth(TN, TM), IT = TN / 32, JT = TM / 32, LA = TN / 8, LX = TM / 8, LOADS = LA + LX;
    static_assert(DEPTH >= 2 && DEPTH <= 4 && 3 * LOADS < 64, "counts of loads under way");
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    unsigned char *ring = s + wave * (DEPTH * BLOCK);
    const Order order(nk, first, wave);
    const int n = order.n;  // this wavefront's steps
    auto issue = [&](int i, int slot) {
        unsigned char *to = ring + slot * BLOCK;
        const int k = order.step(i);
#pragma unroll
        for (int l = 0; l < LA; l++) __builtin_amdgcn_global_load_lds((const PF_AS1 void *)a(l, k), (PF_AS3 void *)(to + 1024 * l), 16, 0, 0);
#pragma unroll
        for (int l = 0; l < LX; l++) __builtin_amdgcn_global_load_lds((const PF_AS1 void *)x(l, k), (PF_AS3 void *)(to + 1024 * (LA + l)), 16, 0, 0);
    };
    unsigned at[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) at[kk] = 128u * (unsigned)(lane & 31) + 16u * (unsigned)((2 * kk + (lane >> 5)) ^ pf_swz(lane & 31));
    f32x16 acc[IT][JT], other[IT][JT];  // (other: the sums before the cut)
    auto clear = [&](f32x16(&c)[IT][JT]) {
#pragma unroll
        for (int i = 0; i < IT; i++)
#pragma unroll
            for (int j = 0; j < JT; j++)
#pragma unroll
                for (int r = 0; r < 16; r++) c[i][j][r] = 0.0f;
    };
    constexpr bool CUT = __is_same(Order, FewEighths);
    clear(acc);
    if constexpr (CUT) clear(other);
    // A step's operands come into registers at once, and the next step of its slot is requested before they are multiplied.  (Reads and their wait in one statement:
    // the compiler would make reads of its own wait for every load under way.)
    pf_u32x4 F[4][IT + JT];
    auto read = [&](int slot) {
        const unsigned lds = (unsigned)(size_t)ring + (unsigned)(slot * BLOCK);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const unsigned p0 = lds + at[2 * h], p1 = lds + at[2 * h + 1];
            pf_u32x4(&F0)[IT + JT] = F[2 * h], (&F1)[IT + JT] = F[2 * h + 1];
            if constexpr (IT + JT == 4)
                asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:4096\n\tds_read_b128 %2, %8 offset:8192\n\tds_read_b128 %3, %8 offset:12288\n\t"
                             "ds_read_b128 %4, %9\n\tds_read_b128 %5, %9 offset:4096\n\tds_read_b128 %6, %9 offset:8192\n\tds_read_b128 %7, %9 offset:12288\n\t"
                             "s_waitcnt lgkmcnt(0)"
                             : "=&v"(F0[0]), "=&v"(F0[1]), "=&v"(F0[2]), "=&v"(F0[IT + JT - 1]), "=&v"(F1[0]), "=&v"(F1[1]), "=&v"(F1[2]), "=&v"(F1[IT + JT - 1])
                             : "v"(p0), "v"(p1)
                             : "memory");
            else if constexpr (IT + JT == 3)
                asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:4096\n\tds_read_b128 %2, %6 offset:8192\n\t"
                             "ds_read_b128 %3, %7\n\tds_read_b128 %4, %7 offset:4096\n\tds_read_b128 %5, %7 offset:8192\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(F0[0]), "=&v"(F0[1]), "=&v"(F0[IT + JT - 1]), "=&v"(F1[0]), "=&v"(F1[1]), "=&v"(F1[IT + JT - 1])
                             : "v"(p0), "v"(p1)
                             : "memory");
            else
                asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:4096\n\tds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(F0[0]), "=&v"(F0[1]), "=&v"(F1[0]), "=&v"(F1[1])
                             : "v"(p0), "v"(p1)
                             : "memory");
        }
    };
    auto multiply = [&](int i_step) {
        if constexpr (CUT)
            if (i_step == order.cut()) {
#pragma unroll
                for (int i = 0; i < IT; i++)
#pragma unroll
                    for (int j = 0; j < JT; j++) other[i][j] = acc[i][j];
                clear(acc);
            }
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
#pragma unroll
            for (int i = 0; i < IT; i++)
#pragma unroll
                for (int j = 0; j < JT; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, F[kk][i]), __builtin_bit_cast(bf16x8, F[kk][IT + j]), acc[i][j], 0, 0, 0);
    };
    for (int i = 0; i < DEPTH && i < n; i++) issue(i, i);
    int slot = 0, i = 0;
    for (; i + DEPTH < n; i++) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * LOADS) : "memory");
        read(slot);
        issue(i + DEPTH, slot);
        multiply(i);
        slot = slot == DEPTH - 1 ? 0 : slot + 1;
    }
    for (; i < n; i++) {
        if (DEPTH >= 4 && n - i == 4)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * LOADS) : "memory");
        else if (DEPTH >= 3 && n - i == 3)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
        else if (n - i == 2)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        read(slot);
        multiply(i);
        slot = slot == DEPTH - 1 ? 0 : slot + 1;
    }
    if constexpr (CUT)
#pragma unroll
        for (int i = 0; i < IT; i++)
#pragma unroll
            for (int j = 0; j < JT; j++) acc[i][j] += other[i][j];
    __syncthreads();  // (the sums' places are another wavefront's ring)
#pragma unroll
    for (int i = 0; i < IT; i++)
#pragma unroll
        for (int j = 0; j < JT; j++)
#pragma unroll
            for (int rq = 0; rq < 4; rq++)
                *(float4 *)(s + 16 * (((wave * IT + i) * JT + j) * FEW_RING_SUMS + 33 * (2 * rq + (lane >> 5)) + (lane & 31))) =
                    make_float4(acc[i][j][4 * rq], acc[i][j][4 * rq + 1], acc[i][j][4 * rq + 2], acc[i][j][4 * rq + 3]);
    __syncthreads();
}
// the sum of rows 4 q .. 4 q + 3 of position p
template <int TN, int TM>
__device__ __forceinline__ float4 few_ring_sum(const unsigned char *s, int p, int q) {
    constexpr int IT = TN / 32, JT = TM / 32;
    static_assert(4 * IT * JT * FEW_RING_SUMS * 16 <= few_ring_lds(TN, TM), "the sums' place");
    float4 v[4];
#pragma unroll
    for (int w = 0; w < 4; w++) v[w] = *(const float4 *)(s + 16 * (((w * IT + (q >> 3)) * JT + (p >> 5)) * FEW_RING_SUMS + 33 * (q & 7) + (p & 31)));
    return make_float4((v[0].x + v[1].x) + (v[2].x + v[3].x), (v[0].y + v[1].y) + (v[2].y + v[3].y), (v[0].z + v[1].z) + (v[2].z + v[3].z),
                       (v[0].w + v[1].w) + (v[2].w + v[3].w));
}
// launches one of the kernels above: workgroups a multiple of 8, LDS beyond 64 KB allowed once a device
#define FEW_RING_DEVICES 64
template <class... P, class... V>
static hipError_t few_ring_go(hipStream_t s, void (*kernel)(P...), bool (&set)[FEW_RING_DEVICES], int lds, int64_t workgroups, V... v) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= FEW_RING_DEVICES) return hipErrorInvalidDevice;
    if (!set[dev]) {
        e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        set[dev] = true;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * ((workgroups + 7) / 8))), dim3(256), lds, s, v...);
    return hipGetLastError();
}
