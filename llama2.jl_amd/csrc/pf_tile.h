// The bf16 tile product of the prompt pass (gfx950 matrix cores), shared by the kernels that run it.
#pragma once

#include "dev_common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    bf16x2 v;
    v.x = (__bf16)a;
    v.y = (__bf16)b;
    return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// Placement of the 16-byte chunks of a 128-byte tile row in LDS.  The LDS has 64 banks of 4 bytes and serves
// 16-byte accesses 16 lanes at a time; lanes read one chunk index of 16 consecutive rows, which the
// exclusive-or with (r >> 1) % 8 sends to the 16 different 16-byte slots of the 256-byte bank row (the row's
// parity picks the half).  With r % 8 instead, rows r and r + 8 collide: half the LDS cycles were conflicts.
__host__ __device__ __forceinline__ int pf_swz(int r) { return (r >> 1) & 7; }

#define PF_AS1 __attribute__((address_space(1)))
#define PF_AS3 __attribute__((address_space(3)))

// Product of bf16 tiles prepared beforehand (32 KB images of 256 weight rows x 64 inputs, 16-byte chunk c of row r at chunk
// index 8 r + (c ^ pf_swz(r))): no arithmetic on the operands.  A workgroup's tile is 256 weight rows
// x 64 JT positions (JT = 4: 256 positions, 64 KB fetched per 64 inputs, half the bytes per product of a 128 x 128 tile; fewer for matrices with too few rows to give
// every CU a 256 x 256 tile, and for blocks of a grouped product), worked on by 8 wavefronts, 4 row groups x 2 position groups, each 64 rows x
// 32 JT positions.  Both operand tiles of a K step travel from global memory
// straight into LDS (16 bytes per lane and load, a wavefront's load filling 1 KB in lane order): the weight
// tile is a linear copy of its 32 KB image, the position tile gets the c ^ pf_swz(r) placement by the choice
// of the address each lane reads.  The loads of step kt + 1 are in flight during the products of step kt, one barrier
// per step, with two LDS stages of up to 72 KB; of the 48 KB stages of JT = 2 three fit, and the loads of step kt + 2 are in
// flight too: where such tiles do not fill the chip a step takes as long as its loads (333 positions x 14 336 rows x 4096
// inputs: 98 us with two stages, 88 with three).
typedef uint32_t pf_u32x4 __attribute__((ext_vector_type(4)));

constexpr int pf_tile_stage(int jt) { return 32768 + 64 * jt * 128; }  // bytes: weight tile, then position tile
constexpr int pf_tile_stages(int jt) { return jt <= 2 ? 3 : 2; }
constexpr int pf_tile_lds(int jt) { return pf_tile_stages(jt) * pf_tile_stage(jt); }

// wtiles: the row group's tiles, K / 64 of them in a row; act: bf16 rows of K elements; s_all: STAGES * pf_tile_stage(JT) bytes of LDS.  row(r) is the
// activation row of the tile's position r; epi(acc, wn, wm, lane) takes the results: a lane holds position
// 32 JT wm + 32 j + lane % 32 and, in register r of tile i, weight row 64 wn + 32 i + 8 (r / 4) + 4 (lane / 32) + r % 4.
template <int JT, int STAGES = pf_tile_stages(JT), class Row, class Epi>
__device__ __forceinline__ void pf_tile_product(const uint16_t *wtiles, const uint16_t *act, int64_t K, uint4 *s_all, Row row, Epi epi) {
    constexpr int STAGE = pf_tile_stage(JT);
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), wn = wave & 3, wm = wave >> 2;
    const int64_t nk = K >> 6;

    // weights: this wavefront copies bytes [4096 wave, +4096) of every tile, 1 KB per load
    const unsigned char *gw = (const unsigned char *)wtiles + wave * 4096 + lane * 16;
    // positions: load i of this wavefront fills chunks 64 (JT wave + i) + lane: row 8 (JT wave + i) + lane / 8,
    // placed chunk lane % 8 = the data chunk (lane % 8) ^ pf_swz(row)
    const unsigned char *gx[JT];
#pragma unroll
    for (int i = 0; i < JT; i++) {
        const int r = 8 * (JT * wave + i) + (lane >> 3);
        gx[i] = (const unsigned char *)(act + row(r) * K + 8 * ((lane & 7) ^ pf_swz(r)));
    }
    // LDS byte offsets of this lane's operands inside a stage: slice kk holds chunk 2 kk + lane / 32 of its rows, and 32 rows further on (4096 bytes, an
    // offset of the read itself) lies the same chunk at the same place of its row
    unsigned aw[4], ax[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
        const unsigned at = 128u * (unsigned)(lane & 31) + 16u * (unsigned)((2 * kk + (lane >> 5)) ^ pf_swz(lane & 31));
        aw[kk] = at + 8192u * (unsigned)wn;
        ax[kk] = at + 32768u + 4096u * (unsigned)(JT * wm);
    }
    const unsigned lds0 = (unsigned)(size_t)s_all;

    f32x16 acc[2][JT];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < JT; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.0f;

    auto issue = [&](int stage) {
        unsigned char *lw = (unsigned char *)s_all + stage * STAGE + wave * 4096;
        unsigned char *lx = (unsigned char *)s_all + stage * STAGE + 32768 + wave * (1024 * JT);
        __builtin_amdgcn_global_load_lds((const PF_AS1 void *)gw, (PF_AS3 void *)lw, 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const PF_AS1 void *)gw, (PF_AS3 void *)lw, 16, 1024, 0);
        __builtin_amdgcn_global_load_lds((const PF_AS1 void *)gw, (PF_AS3 void *)lw, 16, 2048, 0);
        __builtin_amdgcn_global_load_lds((const PF_AS1 void *)gw, (PF_AS3 void *)lw, 16, 3072, 0);
#pragma unroll
        for (int i = 0; i < JT; i++) {
            __builtin_amdgcn_global_load_lds((const PF_AS1 void *)gx[i], (PF_AS3 void *)(lx + 1024 * i), 16, 0, 0);
            gx[i] += 128;
        }
        gw += 32768;
    };

    // The operands of a 16-wide slice (2 weight groups, JT position groups) are read from LDS one slice ahead
    // of the products that use them, into two register sets used in turn, so that a wavefront's LDS latency
    // lies under its own products.  Reads and waits are asm: the compiler then does not make them wait for the
    // copies in flight into the other stage.  Between a PF_READ and the PF_WAIT that retires it the registers
    // of the set hold nothing yet: the set only appears as an operand of those two statements and of the
    // products after the wait (LDS reads complete in order, so lgkmcnt(2 + JT) retires all but the newest set;
    // the build's asm check walks the generated code for any other touch of such a register).
    pf_u32x4 F0[2 + JT], F1[2 + JT];
#define PF_READ(F, KK)                                                                                                                                \
    do {                                                                                                                                              \
        if constexpr (JT == 1)                                                                                                                        \
            asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %3 offset:4096\n\t"                                                                 \
                         "ds_read_b128 %2, %4"                                                                                                        \
                         : "=&v"(F[0]), "=&v"(F[1]), "=&v"(F[2])                                                                                      \
                         : "v"(sb + aw[KK]), "v"(sb + ax[KK])                                                                                         \
                         : "memory");                                                                                                                 \
        else if constexpr (JT == 2)                                                                                                                   \
            asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:4096\n\t"                                                                 \
                         "ds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:4096"                                                                     \
                         : "=&v"(F[0]), "=&v"(F[1]), "=&v"(F[2]), "=&v"(F[3])                                                                         \
                         : "v"(sb + aw[KK]), "v"(sb + ax[KK])                                                                                         \
                         : "memory");                                                                                                                 \
        else if constexpr (JT == 3)                                                                                                                   \
            asm volatile("ds_read_b128 %0, %5\n\tds_read_b128 %1, %5 offset:4096\n\tds_read_b128 %2, %6\n\t"                                          \
                         "ds_read_b128 %3, %6 offset:4096\n\tds_read_b128 %4, %6 offset:8192"                                                         \
                         : "=&v"(F[0]), "=&v"(F[1]), "=&v"(F[2]), "=&v"(F[3]), "=&v"(F[4])                                                            \
                         : "v"(sb + aw[KK]), "v"(sb + ax[KK])                                                                                         \
                         : "memory");                                                                                                                 \
        else if constexpr (JT == 4)                                                                                                                   \
            asm volatile("ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:4096\n\tds_read_b128 %2, %7\n\t"                                          \
                         "ds_read_b128 %3, %7 offset:4096\n\tds_read_b128 %4, %7 offset:8192\n\tds_read_b128 %5, %7 offset:12288"                     \
                         : "=&v"(F[0]), "=&v"(F[1]), "=&v"(F[2]), "=&v"(F[3]), "=&v"(F[4]), "=&v"(F[5])                                               \
                         : "v"(sb + aw[KK]), "v"(sb + ax[KK])                                                                                         \
                         : "memory");                                                                                                                 \
        else if constexpr (JT == 5)                                                                                                                   \
            asm volatile("ds_read_b128 %0, %7\n\tds_read_b128 %1, %7 offset:4096\n\tds_read_b128 %2, %8\n\tds_read_b128 %3, %8 offset:4096\n\t"       \
                         "ds_read_b128 %4, %8 offset:8192\n\tds_read_b128 %5, %8 offset:12288\n\tds_read_b128 %6, %8 offset:16384"                    \
                         : "=&v"(F[0]), "=&v"(F[1]), "=&v"(F[2]), "=&v"(F[3]), "=&v"(F[4]), "=&v"(F[5]), "=&v"(F[6])                                  \
                         : "v"(sb + aw[KK]), "v"(sb + ax[KK])                                                                                         \
                         : "memory");                                                                                                                 \
    } while (0)
    // LAST: nothing newer is in flight
#define PF_WAIT(F, LAST)                                                                                                                              \
    do {                                                                                                                                              \
        if constexpr (JT == 1)                                                                                                                        \
            asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]) : "n"((LAST) ? 0 : 2 + JT) : "memory");                         \
        else if constexpr (JT == 2)                                                                                                                   \
            asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]) : "n"((LAST) ? 0 : 2 + JT) : "memory");             \
        else if constexpr (JT == 3)                                                                                                                   \
            asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]), "+v"(F[4]) : "n"((LAST) ? 0 : 2 + JT) : "memory"); \
        else if constexpr (JT == 4)                                                                                                                   \
            asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]), "+v"(F[4]), "+v"(F[5]) : "n"((LAST) ? 0 : 2 + JT) : "memory");\
        else if constexpr (JT == 5)                                                                                                                   \
            asm volatile("s_waitcnt lgkmcnt(%7)" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]), "+v"(F[4]), "+v"(F[5]), "+v"(F[6]) : "n"((LAST) ? 0 : 2 + JT) : "memory");\
    } while (0)
#define PF_PRODUCTS(F)                                                                                            \
    do {                                                                                                          \
        const bf16x8 W0 = __builtin_bit_cast(bf16x8, F[0]), W1 = __builtin_bit_cast(bf16x8, F[1]);                \
        _Pragma("unroll") for (int j = 0; j < JT; j++) {                                                          \
            const bf16x8 P = __builtin_bit_cast(bf16x8, F[2 + j]);                                                \
            acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(W0, P, acc[0][j], 0, 0, 0);                       \
            acc[1][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(W1, P, acc[1][j], 0, 0, 0);                       \
        }                                                                                                         \
    } while (0)

    // A stage is entered in the middle of the products of the one before: when its last slice's operands are in registers, a
    // wavefront waits for its loads of the next stage, meets the others at the barrier (which says that the next stage is
    // whole and that everyone is done reading this one), sends the loads that overwrite this stage and asks for the next
    // stage's first slice, all before the products of the last slice: the matrix cores do not wait for the barrier or for
    // the first reads behind it.  (2048 positions x 28 672 rows x 4096 inputs in 256 x 256 and 256 x 128 tiles: 473 us with the
    // barrier between the slices of two stages, 439 like this.)
    constexpr int AHEAD = STAGES - 1;  // stages under way
    // this wavefront's loads of the oldest stage under way have landed (NEWER: those of another one may be under way)
#define PF_LANDED(NEWER)                                                                  \
    do {                                                                                  \
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NEWER) ? 4 + JT : 0) : "memory");       \
        __builtin_amdgcn_s_barrier();                                                     \
    } while (0)
    // (the products of F are not to move in front of what stands before this)
#define PF_HERE(F)                                                                                                                \
    do {                                                                                                                          \
        if constexpr (JT == 1)                                                                                                    \
            asm volatile("" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]));                                                                \
        else if constexpr (JT == 2)                                                                                               \
            asm volatile("" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]));                                                    \
        else if constexpr (JT == 3)                                                                                               \
            asm volatile("" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]), "+v"(F[4]));                                        \
        else if constexpr (JT == 4)                                                                                               \
            asm volatile("" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]), "+v"(F[4]), "+v"(F[5]));                            \
        else if constexpr (JT == 5)                                                                                               \
            asm volatile("" : "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3]), "+v"(F[4]), "+v"(F[5]), "+v"(F[6]));                \
    } while (0)
    int stage = 0;
    unsigned sb = lds0;
    for (int i = 0; i < AHEAD && i < nk; i++) issue(i);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (AHEAD < nk) issue(AHEAD);
    PF_READ(F0, 0);
#define PF_SLICES()           \
    do {                      \
        PF_READ(F1, 1);       \
        PF_WAIT(F0, false);   \
        PF_PRODUCTS(F0);      \
        PF_READ(F0, 2);       \
        PF_WAIT(F1, false);   \
        PF_PRODUCTS(F1);      \
        PF_READ(F1, 3);       \
        PF_WAIT(F0, false);   \
        PF_PRODUCTS(F0);      \
        PF_WAIT(F1, true);    \
    } while (0)
#define PF_NEXT_STAGE()                                        \
    do {                                                       \
        stage = stage + 1 == STAGES ? 0 : stage + 1;           \
        sb = lds0 + (unsigned)(stage * STAGE);                 \
        PF_READ(F0, 0);                                        \
        PF_HERE(F1);                                           \
        PF_PRODUCTS(F1);                                       \
    } while (0)
    // (whether a stage is left to load is not asked inside the loops: the last ones have their own)
    int64_t kt = 1;
    for (; kt + AHEAD < nk; kt++) {
        PF_SLICES();
        PF_LANDED(AHEAD == 2);
        issue(stage);
        PF_NEXT_STAGE();
    }
    for (; kt < nk; kt++) {
        PF_SLICES();
        PF_LANDED(false);
        PF_NEXT_STAGE();
    }
    PF_SLICES();
    PF_PRODUCTS(F1);
#undef PF_HERE
#undef PF_LANDED
#undef PF_NEXT_STAGE
#undef PF_SLICES
#undef PF_PRODUCTS
#undef PF_WAIT
#undef PF_READ
    epi(acc, wn, wm, lane);
}

