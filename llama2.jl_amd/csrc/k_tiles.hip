// The many-token products of k_gemm.hip from tile images of the weights (pf_tile.h), bf16 activations: fused epilogues and the
// grouped form for mixtures of experts.
#include "layered_gemm.h"
#include "pf_tile.h"
#include "tiles_plan.h"

// One thread copies a 16-byte chunk of an image: n_mats matrices of `rows` rows, each padded to whole tiles of 256 rows.
__global__ __launch_bounds__(256) void tile_image_kernel(const uint16_t *w, int ld, int64_t rows, int64_t n_chunks, uint16_t *dst) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= n_chunks) return;
    const int64_t nk = ld >> 6, nt_per = (rows + 255) / 256;
    const int within = (int)(idx & 2047), r = within >> 3, c = (within & 7) ^ pf_swz(r);
    const int64_t tile = idx >> 11, kt = tile % nk, ntm = tile / nk, nt = ntm % nt_per, mat = ntm / nt_per;
    const int64_t row = nt * 256 + r;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (row < rows) v = *(const uint4 *)(w + (mat * rows + row) * ld + kt * 64 + 8 * c);
    ((uint4 *)dst)[idx] = v;
}
int64_t k_tile_image_elems(int64_t rows, int ld) { return (rows + 255) / 256 * 256 * ld; }
hipError_t k_tile_image(hipStream_t s, const uint16_t *w, int ld, int64_t rows, int64_t n_mats, uint16_t *dst) {
    if (ld % 64 != 0 || rows < 1) return hipErrorInvalidValue;
    const int64_t n = n_mats * k_tile_image_elems(rows, ld) / 8;
    if ((n + 255) / 256 > 0x7FFFFFFF) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tile_image_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, w, ld, rows, n, dst);
    return hipGetLastError();
}

// 256 rows of the matrix (row group nt of w) x the positions m0 .. of a block of mcount, which starts at row mb
template <int EPI, int JT, int STAGES>
__device__ __forceinline__ void tiles_item(const GemmArgs &a, const uint16_t *w, unsigned nt, int64_t mb, int m0, int mcount, uint4 *s_all) {
    const int64_t n0 = (int64_t)nt * 256;
    pf_tile_product<JT, STAGES>(
        w + (int64_t)nt * (a.ld >> 6) * 16384, (const uint16_t *)a.x, a.ld, s_all,
        [&](int r) {
            const int64_t row = mb + min(m0 + r, mcount - 1);  // (rows past the end repeat the last one; not stored)
            return a.gather ? (int64_t)a.gather[row] : row;
        },
        [&](f32x16(&acc)[2][JT], int wn, int wm, int lane) {
            static_assert(8 * 4 * gemm_epilogue_floats(2, JT) <= STAGES * pf_tile_stage(JT), "the results' place");
            __syncthreads();  // (the operands have all been read)
            float *s = (float *)s_all + (wn + 4 * wm) * gemm_epilogue_floats(2, JT);
            gemm_epilogue<0, EPI, 2, JT>(a, acc, s, mb, m0 + 32 * JT * wm, mcount, n0 + 64 * wn, lane);
        });
}

// a block of up to five units of 64 positions
template <int EPI>
__device__ __forceinline__ void tiles_units(const GemmArgs &a, const uint16_t *w, unsigned nt, int64_t mb, int m0, int mcount, unsigned units, uint4 *s_all) {
    if (units == 5)
        tiles_item<EPI, 5, pf_tile_stages(5)>(a, w, nt, mb, m0, mcount, s_all);
    else if (units == 4)
        tiles_item<EPI, 4, pf_tile_stages(4)>(a, w, nt, mb, m0, mcount, s_all);
    else if (units == 3)
        tiles_item<EPI, 3, pf_tile_stages(3)>(a, w, nt, mb, m0, mcount, s_all);
    else if (units == 2)
        tiles_item<EPI, 2, pf_tile_stages(2)>(a, w, nt, mb, m0, mcount, s_all);
    else
        tiles_item<EPI, 1, pf_tile_stages(1)>(a, w, nt, mb, m0, mcount, s_all);
}

// Items (row group of 256, block of positions) are dealt to the 8 XCDs as contiguous runs: positions fastest in a single
// product, so that workgroups on one weight tile share an L2; row groups fastest in a grouped one, where a block of positions
// is used with one expert's matrix only.
// WHOLE: blocks of 256 positions of a single product, the last items as halves where that pays (tiles_plan); SHARES: its positions in equal shares of up to
// five units; GROUPED: the blocks that a.tiles lists.
enum { TILES_WHOLE = 0, TILES_SHARES = 1, TILES_GROUPED = 2 };
template <int EPI, int MODE>
__global__ __launch_bounds__(512) void tiles_kernel(GemmArgs a, unsigned n_nt, unsigned n_mt, TilesPlan plan) {
    extern __shared__ uint4 s_all[];
    if constexpr (MODE == TILES_WHOLE) {
        const TilesWork work = tiles_work(plan, blockIdx.x);
        if (!work.any) return;
        const int m0 = (int)(work.item % n_mt) * 256;
        if (work.half < 0)
            tiles_item<EPI, 4, pf_tile_stages(4)>(a, a.w, work.item / n_mt, 0, m0, a.M, s_all);
        else if (m0 + 128 * work.half < a.M)
            tiles_item<EPI, 2, pf_tile_stages(2)>(a, a.w, work.item / n_mt, 0, m0 + 128 * work.half, a.M, s_all);
    } else if constexpr (MODE == TILES_SHARES) {
        const TilesBlock k = tiles_block((unsigned)(a.M + TILES_UNIT - 1) / TILES_UNIT, n_mt, plan.n, blockIdx.x);
        if (k.any) tiles_units<EPI>(a, a.w, k.nt, 0, (int)k.at * TILES_UNIT, a.M, k.units, s_all);
    } else {
        const unsigned n_items = (unsigned)a.n_tiles[0] * n_nt, item = tiles_deal(n_items, blockIdx.x);
        if (item >= n_items) return;
        const GemmTile g = a.tiles[item / n_nt];
        tiles_units<EPI>(a, a.w + g.expert * a.expert_stride, item % n_nt, g.row0, 0, g.n, (unsigned)(g.n + TILES_UNIT - 1) / TILES_UNIT, s_all);
    }
}

#define TILES_MAX_DEVICES 64

// n: tiles or items, n_mt: blocks of positions to a row group
template <int EPI, int MODE>
static hipError_t tiles_launch(hipStream_t s, const GemmArgs &a, unsigned n_nt, unsigned n_mt, const TilesPlan &plan) {
    constexpr int lds = std::max(pf_tile_lds(2), pf_tile_lds(MODE == TILES_WHOLE ? 4 : TILES_MAX_UNITS));  // (halves and smaller blocks among them)
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= TILES_MAX_DEVICES) return hipErrorInvalidDevice;
    static bool attr_set[TILES_MAX_DEVICES] = {};
    if (!attr_set[dev]) {
        e = hipFuncSetAttribute((const void *)tiles_kernel<EPI, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        attr_set[dev] = true;
    }
    hipLaunchKernelGGL((tiles_kernel<EPI, MODE>), dim3(tiles_grid(plan)), dim3(512), lds, s, a, n_nt, n_mt, plan);
    return hipGetLastError();
}
// A single product: whole tiles and halves, or shares, whichever are likely through first.  us, whole tiles (of 128 positions where those are fewer than the compute
// units) and shares, 130 / 333 / 640 / 1300 / 2048 positions: 8192 rows x 2048 inputs 36 / 37 / 40 / 76 / 81 and 22 / 24 / 40 / 58 / 81; gated 28 672 x 4096 73 / 118 / 176 /
// 336 / 427 and 73 / 88 / 141 / 322 / 450; 4096 x 1024 25 / 25 / 26 / 28 / 31 and 15 / 16 / 17 / 28 / 31.
template <int EPI>
static hipError_t tiles_single(hipStream_t s, const GemmArgs &a, unsigned n_nt, int n_cu) {
    const unsigned n_mt = (unsigned)((a.M + 255) / 256), units = (unsigned)((a.M + TILES_UNIT - 1) / TILES_UNIT), steps = (unsigned)a.ld >> 6, cu = (unsigned)n_cu;
    const TilesPlan plan = tiles_plan(n_nt * n_mt, true, n_cu);
    const unsigned b = tiles_dense_bound(units, n_nt, steps, cu);
    if (tiles_whole_time(plan, steps, cu) <= tiles_dense_time(units, b, n_nt, steps, cu)) return tiles_launch<EPI, TILES_WHOLE>(s, a, n_nt, n_mt, plan);
    const unsigned blocks = tiles_blocks(units, b);
    return tiles_launch<EPI, TILES_SHARES>(s, a, n_nt, blocks, tiles_plan(n_nt * blocks, false, n_cu));
}

// a.w: the image; otherwise as k_gemm with bf16 activations (ldx == ld)
hipError_t k_tiles(hipStream_t s, const GemmArgs &args, int epi, int n_cu) {
    GemmArgs a = args;
    if (!a.acols) a.acols = a.lda;
    if (!a.w || !a.x || a.n_rows < 1 || a.M < 1 || n_cu < 1 || a.ld % 64 != 0 || a.ldx != a.ld || a.lda % 64 != 0 || a.acols % 64 != 0 ||
        a.acols > a.lda)
        return hipErrorInvalidValue;
    const unsigned n_nt = (unsigned)((a.n_rows + 255) / 256);
    const bool covered = a.outa && a.acols >= a.n_rows && a.acols <= 256 * (int64_t)n_nt;
    const bool pairs = a.outa && a.n_rows % 2 == 0 && 2 * a.acols >= a.n_rows && 2 * a.acols <= 256 * (int64_t)n_nt;
    if (a.tiles) {
        const TilesPlan plan = tiles_plan((unsigned)a.max_tiles * n_nt, false, n_cu);
        if (epi == GE_UP && covered) return tiles_launch<GE_UP, TILES_GROUPED>(s, a, n_nt, 0, plan);
        if (epi == GE_GLU && pairs) return tiles_launch<GE_GLU, TILES_GROUPED>(s, a, n_nt, 0, plan);
        if (epi == GE_STORE && a.outf && a.ldo >= a.n_rows) return tiles_launch<GE_STORE, TILES_GROUPED>(s, a, n_nt, 0, plan);
        return hipErrorInvalidValue;
    }
    if (epi == GE_ACT && covered) return tiles_single<GE_ACT>(s, a, n_nt, n_cu);
    if (epi == GE_GLU && pairs) return tiles_single<GE_GLU>(s, a, n_nt, n_cu);
    return hipErrorInvalidValue;
}
