// One token through a bf16 matrix: a workgroup stages the input vector in LDS behind a fused prologue (norms, expert
// choice), its wavefronts stream whole matrix rows, two at a time, 16 bytes per lane and load, and a fused epilogue writes
// the results.  Activations and sums are fp32 throughout.
#include "rows_dev.h"

template <int PRO, int EPI, int U, int V, bool Y>
__global__ __launch_bounds__(ROWS_THREADS, 4) void rows_kernel(RowsArgs a, RowsPlan pl) {
    extern __shared__ __align__(16) float s_mem[];
    rows_body<PRO, EPI, U, V, Y>(a, pl, blockIdx.x, s_mem);
}
template <int PRO, int EPI, int U, int V, bool Y>
__global__ __launch_bounds__(ROWS_THREADS, 4) void rows_more_kernel(RowsArgs a, RowsPlan pl, RowsMore m) {
    extern __shared__ __align__(16) float s_mem[];
    rows_body<PRO, EPI, U, V, Y>(a, pl, blockIdx.x, s_mem, m);
}

// (a classifier's: see k_rows_keys)
template <int PRO, int EPI, int U, int V, bool Y>
__global__ __launch_bounds__(ROWS_THREADS, 4) void rows_key_kernel(RowsArgs a, RowsPlan pl, RowsKeys k) {
    extern __shared__ __align__(16) float s_mem[];
    rows_body<PRO, EPI, U, V, Y>(a, pl, blockIdx.x, s_mem, RowsMore(), k);
}

#define ROWS_MAX_DEVICES 64

template <int PRO, int EPI, int U, int V, bool Y>
static hipError_t rows_launch(hipStream_t s, const RowsArgs &a, int64_t grid, const RowsMore &m, const RowsKeys &keys) {
    const RowsPlan pl = rows_plan(a, PRO, U, grid);
    const size_t lds = rows_lds(a, PRO, pl.pairs + 1);
    if (lds > ROWS_LDS) return hipErrorInvalidValue;
    const void *fn;
    if constexpr (EPI == RE_RESID_MORE)
        fn = (const void *)rows_more_kernel<PRO, EPI, U, V, Y>;
    else if constexpr (EPI == RE_STORE_KEY)
        fn = (const void *)rows_key_kernel<PRO, EPI, U, V, Y>;
    else
        fn = (const void *)rows_kernel<PRO, EPI, U, V, Y>;
    if (lds > 48 * 1024) {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        if (dev < 0 || dev >= ROWS_MAX_DEVICES) return hipErrorInvalidDevice;
        static bool attr_set[ROWS_MAX_DEVICES] = {};
        if (!attr_set[dev]) {
            e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, ROWS_LDS);
            if (e != hipSuccess) return e;
            attr_set[dev] = true;
        }
    }
    if constexpr (EPI == RE_RESID_MORE)
        hipLaunchKernelGGL((rows_more_kernel<PRO, EPI, U, V, Y>), dim3((unsigned)grid), dim3(ROWS_THREADS), lds, s, a, pl, m);
    else if constexpr (EPI == RE_STORE_KEY)
        hipLaunchKernelGGL((rows_key_kernel<PRO, EPI, U, V, Y>), dim3((unsigned)grid), dim3(ROWS_THREADS), lds, s, a, pl, keys);
    else
        hipLaunchKernelGGL((rows_kernel<PRO, EPI, U, V, Y>), dim3((unsigned)grid), dim3(ROWS_THREADS), lds, s, a, pl);
    return hipGetLastError();
}

// 4 KB of a row at a time where that leaves at least half of the wavefronts' places a step (a 4096 x 4096 matrix: 7.9 us, against
// 8.8 in steps of 1 KB); rows of up to 1024 inputs whole (3072 x 768: 3.5 us against 4.8 in two steps).  A pending update of
// more than 4096 elements takes the registers of the long steps.
static int rows_u(const RowsArgs &a, int pro, int n_cu) {
    const int64_t most = rows_most(a, pro, n_cu);
    if (!(a.y && a.K > 2 * 4 * ROWS_THREADS) && a.ld >= 2048 && rows_steps(a, pro, 4) >= most * ROWS_WAVES / 2) return 4;
    return a.ld > 512 && (rows_steps(a, pro, 2) >= most * ROWS_WAVES / 2 || (a.ld <= 1024 && rows_steps(a, pro, 2) >= n_cu)) ? 2 : 1;
}
int k_rows_workgroups(const RowsArgs &a, int pro, int n_cu) { return (int)rows_grid(a, pro, n_cu, rows_u(a, pro, n_cu)); }

template <int PRO, int EPI, int V, bool Y>
static hipError_t rows_split(hipStream_t s, const RowsArgs &a, int n_cu, const RowsMore &m, const RowsKeys &keys) {
    const int u = rows_u(a, PRO, n_cu);
    const int64_t grid = rows_grid(a, PRO, n_cu, u);
    if constexpr (!(Y && V > 2))
        if (u == 4) return rows_launch<PRO, EPI, 4, V, Y>(s, a, grid, m, keys);
    if (u == 2) return rows_launch<PRO, EPI, 2, V, Y>(s, a, grid, m, keys);
    return rows_launch<PRO, EPI, 1, V, Y>(s, a, grid, m, keys);
}

// the vector's registers: two steps for up to 4096 elements behind a norm, four for more; eight for one that is staged as it is
template <int PRO, int EPI>
static hipError_t rows_pick(hipStream_t s, const RowsArgs &a, int n_cu, const RowsMore &m, const RowsKeys &keys) {
    if constexpr (PRO == RP_PLAIN || PRO == RP_DOWN) {
        return rows_split<PRO, EPI, 8, false>(s, a, n_cu, m, keys);
    } else if constexpr (PRO == RP_HEADNORM) {
        return a.K <= 2 * 4 * ROWS_THREADS ? rows_split<PRO, EPI, 2, false>(s, a, n_cu, m, keys) : rows_split<PRO, EPI, 4, false>(s, a, n_cu, m, keys);
    } else {
        const bool few = a.K <= 2 * 4 * ROWS_THREADS;
        if constexpr (PRO == RP_NORM && (EPI == RE_STORE || EPI == RE_STORE_GLU || EPI == RE_STORE_KEY)) {
            if (a.y) return few ? rows_split<PRO, EPI, 2, true>(s, a, n_cu, m, keys) : rows_split<PRO, EPI, 4, true>(s, a, n_cu, m, keys);
        }
        if (a.y) return hipErrorInvalidValue;
        return few ? rows_split<PRO, EPI, 2, false>(s, a, n_cu, m, keys) : rows_split<PRO, EPI, 4, false>(s, a, n_cu, m, keys);
    }
}

hipError_t k_rows(hipStream_t s, const RowsArgs &a, int pro, int epi, int n_cu, const RowsMore &more) {
    if (!a.w || !a.x || !a.out || a.n_rows < 1 || a.n_rows > 0x7FFFFFFF || a.ld % 64 != 0 || a.K > a.ld || a.K < 1) return hipErrorInvalidValue;
    if ((pro == RP_UP || pro == RP_DOWN) && (!a.z || !a.sel || a.n_experts < 1 || a.n_experts > ROWS_MAX_EXPERTS || a.top < 1 || a.top > ROWS_MAX_TOP ||
                                             a.top > a.n_experts || a.n_experts * a.rows_each > 0x7FFFFFFF))
        return hipErrorInvalidValue;
    if ((epi == RE_GLU && a.n_rows % 2 != 0) || (epi == RE_STORE_GLU && (a.n_rows % 2 != 0 || a.glu_from % 2 != 0 || !a.out2)))
        return hipErrorInvalidValue;
    RowsMore m = more;
    if (m.stride || m.plus || m.plus2) {
        if (epi != RE_RESID || (m.stride && pro == RP_DOWN)) return hipErrorInvalidValue;
        epi = RE_RESID_MORE;
    }
    if (!m.stride) m.stride = a.ld;
#define GO(P, E) \
    if (pro == P && epi == E) return rows_pick<P, E>(s, a, n_cu, m, RowsKeys())
    GO(RP_NORM, RE_STORE);
    GO(RP_NORM, RE_ACT);
    GO(RP_PLAIN, RE_STORE);
    GO(RP_PLAIN, RE_RESID);
    GO(RP_PLAIN, RE_EMBED);
    GO(RP_UP, RE_UP);
    GO(RP_NORM, RE_GLU);
    GO(RP_NORM, RE_STORE_GLU);
    GO(RP_UP, RE_GLU);
    GO(RP_DOWN, RE_RESID);
    GO(RP_PLAIN, RE_RESID_MORE);
    GO(RP_DOWN, RE_RESID_MORE);
    GO(RP_HEADNORM, RE_RESID_MORE);
    GO(RP_HEADNORM, RE_RESID);
#undef GO
    return hipErrorInvalidValue;
}

hipError_t k_rows_keys(hipStream_t s, const RowsArgs &a, int n_cu, const RowsKeys &keys) {
    if (!a.w || !a.x || !a.out || a.n_rows < 1 || a.n_rows > 0x7FFFFFFF || a.ld % 64 != 0 || a.K > a.ld || a.K < 1 || !keys.keys || !keys.ctl || !keys.next) return hipErrorInvalidValue;
    return rows_pick<RP_NORM, RE_STORE_KEY>(s, a, n_cu, RowsMore(), keys);
}
