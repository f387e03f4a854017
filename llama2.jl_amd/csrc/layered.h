// Layered models: kernels and launchers of the mechanisms a layer can be composed of (k_rows.hip, k_delta.hip,
// k_window.hip, k_latent.hip, k_gemm.hip).  Matrices are bf16 rows of `ld` elements (a multiple of 64, zero from K on); vectors,
// caches and recurrent state are fp32.
#pragma once

#include "l2h_internal.h"
#include "tiles_plan.h"

struct LMat {
    uint16_t *w = nullptr;
    int64_t rows = 0;
    int K = 0, ld = 0;
    // tile image for the prompt pass (k_tiles.hip), or nullptr; elements of one matrix where several are stacked
    uint16_t *image = nullptr;
    int64_t image_stride = 0;
};
static inline int pad64(int64_t n) { return (int)((n + 63) / 64 * 64); }

static inline int pad4(int64_t n) { return (int)((n + 3) / 4 * 4); }

enum { LACT_GELU_ERF = 0, LACT_RELU2 = 1, LACT_GELU_TANH = 2, LACT_RELU = 3, LACT_SILU = 4 };
// how a router's logits become weights: a sigmoid each, on the expert's input, or the softmax over the chosen, on its output
enum { LROUTE_SIGMOID_IN = 0, LROUTE_SOFTMAX_OUT = 1 };

// ---- one token: matrix x vector with a fused prologue and epilogue (k_rows.hip) ---------------------------------
// prologues: what the vector in LDS is
//   RP_PLAIN    x
//   RP_NORM     rmsnorm(x) * normw; with y set, x first takes the pending update x += mult * rmsnorm(y) * yw, which
//               workgroup 0 also writes to x_out
//   RP_UP       as RP_NORM; the rows are those of the `top` experts with the largest z, `rows_each` rows each
//   RP_DOWN     x holds `top` vectors of K elements; every output row sums the chosen experts' rows
//   RP_HEADNORM x[h * hv + j] * rms over the head's hv elements (from partial sums of squares) * normw[j] * gate[...]
enum { RP_PLAIN = 0, RP_NORM = 1, RP_UP = 2, RP_DOWN = 3, RP_HEADNORM = 4 };
// epilogues: RE_STORE v; RE_RESID resid + mult * v; RE_ACT act(v); RE_UP act(score * v) or score * act(v) with the expert's score;
// RE_EMBED act(v) * emb[row]; RE_GLU rows 2 i and 2 i + 1 give out[i] = act(v) * v', with the
// expert's score behind RP_UP; RE_STORE_GLU stores rows below glu_from and treats the others so, into out2; RE_STORE_AGENT v, past the
// caches of the storing workgroup; RE_RESID_MORE as RE_RESID, with a RowsMore (k_rows takes it where one of its fields is set); RE_STORE_KEY v, and a
// workgroup's largest (k_rows_keys)
enum { RE_STORE = 0, RE_RESID = 1, RE_ACT = 2, RE_UP = 3, RE_EMBED = 4, RE_GLU = 5, RE_STORE_GLU = 6, RE_STORE_AGENT = 7, RE_RESID_MORE = 8, RE_STORE_KEY = 9 };
struct RowsArgs {
    const uint16_t *w = nullptr;
    int ld = 0, K = 0;
    int64_t n_rows = 0;
    const float *x = nullptr;
    float *out = nullptr;
    float mult = 1.0f, eps = 0.0f;
    const float *normw = nullptr;
    const float *y = nullptr, *yw = nullptr;
    float *x_out = nullptr;
    const float *resid = nullptr;
    int act = 0;
    int64_t glu_from = 0;
    float *out2 = nullptr;
    const float *z = nullptr, *z_bias = nullptr;  // router logits
    int n_experts = 0, top = 0, route = 0;
    int64_t rows_each = 0;
    const float *ssq = nullptr, *gate = nullptr;  // RP_HEADNORM
    int hv = 0, n_split = 0;
    const uint16_t *emb = nullptr;  // RE_EMBED
    int32_t *sel = nullptr;         // RP_UP leaves the chosen experts there, RP_DOWN finds them
};
// What few products of a residual have.  Apart, for the sake of the others: with these fields and their branches in every launch a token of Vudelix took 1 % longer
// (width 768, 4 layers: 170.6 us against 169.2).
struct RowsMore {
    int64_t stride = 0;                             // from row to row (0: ld); not for RP_DOWN
    const float *plus = nullptr, *plus2 = nullptr;  // vectors added to the sum, one after the other
};
hipError_t k_rows(hipStream_t s, const RowsArgs &a, int pro, int epi, int n_cu, const RowsMore &more = RowsMore());
// A step's classifier: as RP_NORM, RE_STORE; each of its k_rows_workgroups() workgroups also leaves the key (argmax_key) of its first largest row, and the
// first of them `ctl` in `next`, marked: what the next step's k_step_begin picks the token from.
struct RowsKeys {
    unsigned long long *keys = nullptr;
    const DecodeCtl *ctl = nullptr;
    DecodeCtl *next = nullptr;
};
int k_rows_workgroups(const RowsArgs &a, int pro, int n_cu);
hipError_t k_rows_keys(hipStream_t s, const RowsArgs &a, int n_cu, const RowsKeys &keys);

// ---- many tokens: C[m][n] = sum_k X[m][k] W[n][k] (k_gemm.hip) ---------------------------------------------------
// activations are bf16 (prec 0) or fp32 (prec 1: fp32 products on the matrix cores); ldx a multiple of 64, zero from K on
enum {
    GE_STORE = 0,   // outf = v
    GE_RESID = 1,   // outf += mult * v
    GE_ACT = 2,     // outa = act(v)
    GE_UP = 3,      // outa = act(row_scale[m] * v), or row_scale[m] * act(v) without scale_in
    GE_EMBED = 4,   // outa = act(v) * embedding element
    GE_DECAY = 5,   // outf = -rate[n / hd] * softplus(v + bias[n]): the logarithm of a decay
    GE_SIGMOID = 6, // outf = sigmoid(v)
    GE_GLU = 7      // columns 2 i and 2 i + 1 give outa[i] = act(v) * v'; with row_scale as GE_UP, on both factors or on the result
};
struct GemmTile {  // a block of rows of a grouped product
    int32_t expert, row0, n;
};
struct GemmArgs {
    const uint16_t *w = nullptr;
    int64_t n_rows = 0;
    int ld = 0;
    const void *x = nullptr;
    int64_t ldx = 0;
    int M = 0;
    float *outf = nullptr;
    int64_t ldo = 0;
    void *outa = nullptr;  // activation-typed, columns up to acols (0: lda) are zeroed from the last result on
    int64_t lda = 0, acols = 0;
    int scale_in = 1;
    float mult = 1.0f;
    int act = 0;
    const float *row_scale = nullptr;
    const uint16_t *emb = nullptr;
    int64_t emb_ld = 0;
    const int32_t *tokens = nullptr;
    const float *rate = nullptr, *bias = nullptr;
    int hd = 1;
    // grouped form: tiles lists blocks of rows, each with its own matrix w + expert * expert_stride
    const GemmTile *tiles = nullptr;
    const int32_t *n_tiles = nullptr;
    int max_tiles = 0;
    int64_t expert_stride = 0;
    int matrices = 0, rows_each = 0;  // how many there are; rows of one on average
    bool few = false;   // to k_few, whatever k_few_pays says
    const int32_t *gather = nullptr;  // row of x for each row of the product
    // where workgroups that share a block of results leave their sums (FEW_PART_FLOATS), and how many are through with each (FEW_PART_ITEMS, zero between
    // launches); without, nothing is shared out
    float *part = nullptr;
    unsigned *arrived = nullptr;
};
#define L_GEMM_TILE 128  // rows of a block for k_gemm
hipError_t k_gemm(hipStream_t s, const GemmArgs &a, int prec, int epi);
// The same for few rows or positions (k_few.hip), which k_gemm hands on to where that is the faster way; cols: columns the epilogue
// covers.  Distinct matrices one after the other:
//
// bf16, the time of k_gemm's own tiles over that of k_few.  Grouped, up to 48 positions a matrix (8 and 16 matrices of 256 to 2048 inputs, at 8 and 32 1.8 to 2.6 and 1.7 to
// 2.3), and up to 60 where there are few blocks of 64 rows, for longer loops more: 60 positions each of 64, 256, 512, 1024 and 2048 inputs, 128 blocks 1.0 to 1.1, 1.3, 1.6, 2.0 and 2.4, 256
// 0.85 to 0.9, 1.1, 1.2, 1.4 to 1.5 and 1.6, 512 0.6, 0.8, 0.8 to 1.0, 0.9 to 1.1 and 1.0 to 1.2, 1024 0.4, 0.5, 0.6 to 0.7, 0.7 to 0.8 and 0.9 to 1.1.  Plain, up to 64 positions, up to 128 of at
// least 768 inputs (1.0 to 2.0, up to 32 000 rows; 65 to 128 of fewer inputs in more than 256 tiles of 64 x 64 0.6 to 0.9), otherwise where such tiles are at most 256
// (1.0 to 1.9), or 768 of at least 2048 inputs: 288 tiles 1.6, 512 1.3, 768 1.1, 1500 0.9; of 512 inputs 512 tiles 0.8.
//
// fp32, k_few's time over that of the tiles, at 256 to 4096 inputs.  Plain, up to 8 positions (0.3 to 0.97) and up to 2^17 results, 2^18 of up to 16 positions: of 17
// positions and more 0.5 to 0.95 up to 2^16.5 results, 0.65 to 1.01 at 2^17, 0.95 to 1.34 at 2^17.5, 0.96 to 1.77 at 2^18, 1.2 to 2.1 at 2^20; of 9 to 12 positions 0.82 to
// 1.08 beyond 2^18, where the tiles, whose sums are nearer to 64 bits (of 256 inputs 0.9e-7 against 1.5e-7, of 4096 1.4e-7 and 4.0e-7), take them all the same; of 16 0.99 to
// 1.15 at 2^18.  (With an activation behind them, from 2^17 to 2^18.3 results: up to 512 inputs 0.7 to 1.0, a microsecond, for the same reason.)  Grouped, up to 64 positions a matrix and 2^18
// results: 8, 16, 32 and 64 positions each 0.4 to 0.99 up to 2^17, 0.75 to 1.27 at 2^18, 0.93 to 1.66 at 2^19; of 2 and 4 each 0.9 to 1.2; of 100 each 1.13 to 1.6, of 128
// 1.2 to 1.9, of 512 1.2 to 1.9 up to 2^17.
// tiles of a product that workgroups share out, at most, and their sums
#define FEW_PART_ITEMS 256
#define FEW_PART_FLOATS (FEW_PART_ITEMS * 64 * 64)
#define L_FEW_M 128
#define L_FEW_M_F32 8
#define L_FEW_EACH 48
#define L_FEW_EACH_MOST 60
#define L_FEW_EACH_F32 64
#define L_FEW_TILES 256
#define L_FEW_RESULTS_F32 131072
inline int64_t few_blocks(const GemmArgs &a, int64_t cols) { return a.matrices * ((cols + 63) / 64); }  // of 64 rows
inline bool k_few_pays(const GemmArgs &a, int prec, int64_t cols) {
    if (prec) return a.M <= L_FEW_M_F32 || (a.M * cols <= (a.tiles || a.M <= 16 ? 2 : 1) * L_FEW_RESULTS_F32 && (!a.tiles || a.rows_each <= L_FEW_EACH_F32));
    if (a.few) return true;
    if (a.tiles) return a.rows_each <= L_FEW_EACH || (a.rows_each <= L_FEW_EACH_MOST && few_blocks(a, cols) <= (a.ld >= 2048 ? 2 * L_FEW_TILES : a.ld >= 256 ? L_FEW_TILES : L_FEW_TILES / 2));
    return a.M <= (a.ld >= 768 ? L_FEW_M : L_FEW_M / 2) || ((cols + 63) / 64) * ((a.M + 63) / 64) <= (a.ld >= 2048 ? 3 : 1) * L_FEW_TILES;
}
hipError_t k_few(hipStream_t s, const GemmArgs &a, int prec, int epi, int64_t cols);
// Experts' products of a bf16 prompt that have a tile image: k_few from the plain rows where the image's row groups of 256 are too few for the compute units, and the inputs or positions not so few
// that a tile is all prologue and epilogue (60 and 128 positions each, 64 groups of 64 inputs 5.4, 6.2 and 7.6, 11.8, of 256 7.7, 8.2 and 9.9, 13.3; 16 groups 4.4, 5.3 and 3.9, 5.0).  us, k_tiles
// and k_few, 16, 48 and 83 positions an expert: 8 of 512 x 512 (16 groups) 7.2, 9.9, 11.0 and 4.0, 6.1, 7.3; 32 of 512 x 1024 (64) 16.6, 19.7, 21.6 and 9.5, 14.2, 16.6; 8 of
// 1792 x 3584 (56) 42, 51, 54 and 21, 36, 38; 128 each 1.3 to 1.5 times; 16 of 2048 x 4096 (128) 56, 64, 72 and 48, 64, 85; 32 of 1024 x 2048 (128) 31, 35, 38 and 28, 36, 47; 16 of
// 2048 x 1024 (128) 17.5, 20.6, 23.3 and 17.2, 23.0, 29.4; 16 of 4096 x 2048 (256) 49, 52, 57 and 51, 70, 95.
inline bool k_few_experts_pays(int experts, int64_t rows, int ld, int rows_each) {
    const int64_t groups = experts * ((rows + 255) / 256);
    return (groups <= 64 && rows_each <= 128 && (groups <= 16 || rows_each <= 40 || ld >= 512)) || (groups <= 128 && rows_each <= 32 && ld >= 2048);
}
// A plain product (GE_STORE, GE_RESID) that the library would take: k_few where tiles of 64 x 64 are at most one a compute unit and its inputs few enough.  us, the library
// with positions in whole groups of 128 and k_few, 130, 256, 333 and 500 positions: 1024 x 1024 5.5, 5.4, 6.5, 6.5 and 4.5, 4.6, 5.7, 5.8; 2048 x 2048 10.1, 10.1, 12.6, 12.8 and 8.1, 9.1,
// 10.3, 11.5; 1024 x 4096 12.0, 12.0, 15.1, 15.7 and 10.3, 11.2, 12.0, 15.1; 4096 x 4096 22.9, 22.8 and 18.3, 23.0, but 333 (384 tiles) 24.9 and 32.5; 2048 x 6144 23.2, 23.2, 27.5, 27.3 and
// 17.7, 21.1, 29.0, 31.7; 6144 x 2048, 130 (288) 16.0 and 20.5.  More than 512 positions only of a router: 2048 of 32 x 2048 6.8 and 5.4, but of 256 x 2048 8.8 and 13.0.
// Few rows of many inputs go better in more shares than eight: 128 x 3072, 256 6.0 and 6.8, 128 x 4096 6.6 and 7.8, 512 x 4096, 256 and 512 8.1, 10.0 and 8.6, 11.2, but 128 x 2048 5.4 and 5.4, 512 x 3072
// 7.2, 8.4 and 6.6, 7.0, 768 x 4096 11.9, 14.9 and 10.3, 14.1.  Of 256 inputs, 130, 256 and 512, 1344 rows 4.5 (256), 5.2 (512) and 4.0, 5.9; 2048 4.6, 4.7, 5.3 and 4.1, 4.2, 6.2; 4096 5.3, 5.3 and 5.8, 6.2 (tiles of
// 32 rows up to 256, where few_plan takes them).  Not so where embedding rows come behind (a.emb), another launch after the library's: 256 x 4096, 333 positions 11.4 + 5.0
// and 13.3.
inline bool k_few_plain_pays(const GemmArgs &a) {
    const int64_t positions = (a.M + 63) / 64, small = (a.n_rows + 31) / 32 * positions;
    const bool tiles = (a.M <= 512 || a.n_rows <= 32) && (a.n_rows + 63) / 64 * positions <= L_FEW_TILES && (a.ld <= 4096 || a.M <= 256);
    if (a.emb) return tiles;
    return tiles && (a.ld <= 2048 || a.n_rows <= 32 || 6 * a.n_rows >= a.ld) && (a.ld < 256 || a.ld >= 384 || small <= L_FEW_TILES);
}

// the same from a tile image (k_tiles.hip): GE_ACT, GE_GLU, and GE_UP / GE_GLU / GE_STORE in the grouped form; bf16 activations
hipError_t k_tiles(hipStream_t s, const GemmArgs &a, int epi, int n_cu);
int64_t k_tile_image_elems(int64_t rows, int ld);
hipError_t k_tile_image(hipStream_t s, const uint16_t *w, int ld, int64_t rows, int64_t n_mats, uint16_t *dst);
// outa[m][n] = act(v[m][n]) * embedding element, for products that the library has stored as fp32
hipError_t k_embed_rows(hipStream_t s, const float *v, int M, int N, int act, const uint16_t *emb, int64_t emb_ld,
                        const int32_t *tokens, void *outa, int64_t lda, int prec);

// rows of x (fp32, stride K): [x += mult * rmsnorm(y) * yw;] outa = rmsnorm(x) * w, or x itself with w == nullptr; with
// `gather`, row r of the result is row gather[r] of x
hipError_t k_norm_rows(hipStream_t s, float *x, int K, int M, const float *w, float eps, const float *y, const float *yw,
                       float mult, const int32_t *gather, void *outa, int64_t lda, int prec);

// ---- mixture of experts, many tokens (k_gemm.hip) ----------------------------------------------------------------
// z[M][ldz] (+ bias) -> choice[M][top], score[M][top]; then the grouping: slot_row / slot_scale per slot (slots of an expert are
// consecutive), slot_of[M][top], tiles
hipError_t k_route(hipStream_t s, const float *z, int64_t ldz, const float *bias, int M, int E, int top, int kind, int32_t *choice,
                   float *score);
hipError_t k_group(hipStream_t s, const int32_t *choice, const float *score, int M, int E, int top, int32_t *slot_row,
                   float *slot_scale, int32_t *slot_of, GemmTile *tiles, int32_t *n_tiles, int tile_rows);
// with a list of blocks for each of two products from tile images, by rule[p] (tiles_plan.h): tiles[p], n_tiles[p]
hipError_t k_group_images(hipStream_t s, const int32_t *choice, const float *score, int M, int E, int top, int32_t *slot_row, float *slot_scale,
                          int32_t *slot_of, GemmTile *const tiles[2], int32_t *n_tiles, const TilesRule rule[2]);
// x[m] += mult * sum_k y[slot_of[m][k]]
hipError_t k_gather_add(hipStream_t s, float *x, const float *y, const int32_t *slot_of, int M, int top, int K, float mult);
// x[m] += a[m] + b, a or not
hipError_t k_stream_add(hipStream_t s, float *x, const float *a, const float *b, int M, int K);

// ---- gated delta rule with one decay per key channel (k_delta.hip) -----------------------------------------------
// The projected row of a token: q [G D] | k [G D] | v [H V] | beta logits [H] | decay factor [ra] | gate factor [rg].
struct DeltaShape {
    int H, G, D, V, taps, ra, rg;
    float eps;
    __host__ __device__ int channels() const { return 2 * G * D + H * V; }
    __host__ __device__ int off_b() const { return channels(); }
    __host__ __device__ int off_a() const { return channels() + H; }
    __host__ __device__ int off_g() const { return channels() + H + ra; }
    __host__ __device__ int n_in() const { return channels() + H + ra + rg; }
};
#define L_DELTA_COLS 32  // value columns per workgroup of the one-token kernel
static inline int delta_splits(int V) { return (V + L_DELTA_COLS - 1) / L_DELTA_COLS; }
struct DeltaWeights {
    const float *conv;  // [taps][channels], the current token's tap last
    const float *rate, *bias;  // [H], [H D]
    const uint16_t *a2, *g2;
    int lda2, ldg2;
};
// ring: [taps][channels], slot t % taps holds token t's projected channels; state: [H][D][V]
hipError_t k_delta_step(hipStream_t s, const DeltaShape &d, const DeltaWeights &w, const float *in, float *ring, float *state,
                        const DecodeCtl *ctl, float *o, float *ssq, float *gate);
// convolution, silu, unit vectors, beta: raw[M][ldr] -> qkv[M][channels], kq[M][G] (= k . q; or nullptr), beta[M][H], and the two low-rank
// factors as activations
hipError_t k_delta_prepare(hipStream_t s, const DeltaShape &d, const float *conv, const float *raw, int64_t ldr, const float *ring,
                           int M, int pos0, float *qkv, float *kq, float *beta, void *fa, int64_t lfa, void *fg, int64_t lfg,
                           int prec);
// the recurrence over M tokens, logarithms of the decays in lg[M][H D]; o[M][H V]; then the ring takes the last tokens
hipError_t k_delta_scan(hipStream_t s, const DeltaShape &d, const float *qkv, const float *kq, const float *beta, const float *lg,
                        float *state, int M, int pos0, float *o);
// the same in chunks on the matrix cores, with k_head_norm_rows behind it; scratch: rec and the rows of o as delta_plan.h says
hipError_t k_delta_walk(hipStream_t s, const DeltaShape &d, const float *qkv, const float *beta, const float *lg, float *state, int M, int pos0, float *rec,
                        int64_t rec_floats, float *o, const float *gate, const float *normw, void *outa, int64_t lda, int prec);
// Tokens from which the chunked form is used.  Prompts of 24, 40, 48 and 64 through three layers, us, the scan and chunks: 16 heads of 128 x 128 464 and 488, 540 and 549, 553
// and 549, 587 and 560; 16 of 64 x 64 345 and 362, 370 and 369, 379 and 373, 394 and 375; 8 of 256 x 256 433 and 465, 479 and 487, 493 and 494, 529 and 499.
#define L_DELTA_WALK_MIN 48
hipError_t k_delta_ring(hipStream_t s, const DeltaShape &d, const float *raw, int64_t ldr, float *ring, int M, int pos0);
// outa[m][h V + j] = o * rms over the head * normw[j] * gate
hipError_t k_head_norm_rows(hipStream_t s, const float *o, const float *gate, const float *normw, int M, int H, int V, float eps,
                            void *outa, int64_t lda, int prec);

// ---- attention over a sliding window (k_window.hip) --------------------------------------------------------------
// The projected row of a token: q [H D] | k [G D] | v [G V] | gate logits [H].
struct WindowShape {
    int H, G, D, V, window, rot, gated, qk_norm;  // rot: rotated dimensions
    int rot_half;                                 // pairs i, i + rot / 2 instead of 2i, 2i+1
    float scale, eps;
    int seq_len;
    __host__ __device__ int Dp() const { return (D + 3) / 4 * 4; }  // key elements per cache row: kc[G][Dp / 4][seq_len][4]; vc[G][seq_len][V]
    __host__ __device__ int off_k() const { return H * D; }
    __host__ __device__ int off_v() const { return H * D + G * D; }
    __host__ __device__ int off_g() const { return H * D + G * D + G * V; }
    __host__ __device__ int n_in() const { return H * D + G * D + G * V + (gated ? H : 0); }
};
#define L_WIN_SPLIT 64  // keys per workgroup of the one-token kernel (a lane each)
static inline int window_splits(const WindowShape &w) { return (std::min(w.window, w.seq_len) + L_WIN_SPLIT - 1) / L_WIN_SPLIT; }
hipError_t k_window_step(hipStream_t s, const WindowShape &w, const float *freq, const float *in, float *kc, float *vc,
                         const DecodeCtl *ctl, float *part, float *out);
static inline int64_t window_part_floats(const WindowShape &w) { return (int64_t)w.H * window_splits(w) * (w.V + 2); }
// rotation + norm of q and k, cache append; q as fp32 [M][H D] (qf) or bf16 [M][H hs] (qb, zero beyond D)
hipError_t k_window_prepare(hipStream_t s, const WindowShape &w, const float *freq, const float *raw, int64_t ldr, float *kc,
                            float *vc, int M, int pos0, float *qf, uint16_t *qb, int hs);
// fp32 attention of M queries over the cache, output gate included
hipError_t k_window_rows(hipStream_t s, const WindowShape &w, const float *qf, const float *raw, int64_t ldr, const float *kc,
                         const float *vc, int M, int pos0, void *outa, int64_t lda, int prec);

// ---- attention over a cached latent (k_latent.hip) ---------------------------------------------------------------
// The projected row of a token: query latent [Q] | key/value latent [C] and rotated key part [R] | gates [H V], each part
// from a multiple of four on.  The cache holds a row of ld() floats per position: the normed latent, zeros up to Cp, the
// rotated part, zeros.  A head's key is [k_up c | rotated part], its value v_up c; one token's queries are taken through
// k_up^T instead, so that scores and values are formed on the cached rows, which all heads share, and v_up is applied to the
// result.  ukv: the rows of k_up (H D), then of v_up (H V), of C inputs.
struct LatentShape {
    int H, D, R, V, C, Q, rot, rot_half, gated;
    float scale, eps;
    int seq_len;
    __host__ __device__ int Cp() const { return (C + 15) / 16 * 16; }
    __host__ __device__ int Rp() const { return (R + 15) / 16 * 16; }
    __host__ __device__ int ld() const { return Cp() + Rp(); }
    __host__ __device__ int hq() const { return D + R; }
    __host__ __device__ int off_kv() const { return (Q + 3) / 4 * 4; }
    __host__ __device__ int off_g() const { return (off_kv() + C + R + 3) / 4 * 4; }
    __host__ __device__ int n_in() const { return (off_g() + (gated ? H * V : 0) + 3) / 4 * 4; }
};
#define L_LATENT_MAX_RANK 1024
#define L_LATENT_BLOCK 128  // tokens whose queries go through k_up^T at a time
#define L_LATENT_SMALL 16   // up to so many tokens of a prompt go that way, more through their heads' own keys and values
#define L_LATENT_SPLITS 128
// workgroups that share the keys of one block of 16 (token, head) columns
static inline int latent_splits(int64_t cols) {
    return (int)std::min<int64_t>(L_LATENT_SPLITS, std::max<int64_t>(1, 512 / ((cols + 15) / 16)));
}
static inline int64_t latent_part_floats(const LatentShape &w, int64_t cols) { return cols * latent_splits(cols) * (w.Cp() + 4); }
// raw[M][ldr] -> cache rows pos0 .., and the normed query latent as activations cq[M][lcq]
hipError_t k_latent_prepare(hipStream_t s, const LatentShape &w, const float *qnorm, const float *kvnorm, const float *freq,
                            const float *raw, int64_t ldr, float *cache, int M, int pos0, void *cq, int64_t lcq, int prec);
// q[M][H hq] -> qa[M H][ld]: rotated, the unrotated part through k_up^T.  With ctl the position is the decode step's and the
// token's own cache row is made from its projected row `in` by the same launch.
hipError_t k_latent_query(hipStream_t s, const LatentShape &w, const float *freq, const float *q, const uint16_t *ukv, int ldu,
                          float *qa, int M, int pos0, const DecodeCtl *ctl, const float *in, const float *kvnorm, float *cache);
// partial softmax sums of the cached rows, part: latent_part_floats(w, M H)
hipError_t k_latent_attend(hipStream_t s, const LatentShape &w, const float *qa, const float *cache, float *part, int M, int pos0,
                           const DecodeCtl *ctl);
// joins them, applies v_up and the gates raw[m][ldr]: outa[m][h V + e], columns H V .. cols - 1 zeroed
hipError_t k_latent_value(hipStream_t s, const LatentShape &w, const float *part, const uint16_t *ukv, int ldu, const float *raw,
                          int64_t ldr, int M, void *outa, int64_t lda, int64_t cols, int prec, const DecodeCtl *ctl);
// for the matrix-core attention: rotated queries as bf16 [M][H hs], cached latents n rows from pos0 as activations [n][lda]
hipError_t k_latent_heads(hipStream_t s, const LatentShape &w, const float *freq, const float *q, uint16_t *qb, int hs, int M, int pos0);
hipError_t k_latent_rows(hipStream_t s, const LatentShape &w, const float *cache, int pos0, int n, uint16_t *outa, int64_t lda);

// ---- a decode step's latent attention and feed-forward in shared launches (k_step.hip) ----------------------------
#define L_STEP_RANK 512   // elements of the cached latent at most (a lane's eight; a thread of 512 each)
#define L_STEP_ROT 64
#define L_STEP_HEAD 128   // elements of a head's key, without its rotated part, and of its value
#define L_STEP_RUN 32     // keys of a workgroup, at least ...
#define L_STEP_SPLITS 16  // ... and workgroups of a head, at most
// Longest sequence, of fewer than eight heads half of it (a workgroup's keys go one batch of 32 after the other).  Microseconds a token in
// launches of their own and shared, at positions 100, 1000, 2000, 4000: 16 heads, width 2048, 4 layers (6 runs): 320 330 345 364, 254 305 324
// 355; 32 heads, width 4096, 2 layers: 246 252 257 266, 207 236 239 255; 9 heads, width 1152, 2 layers: 96 97 101 105, 80 96 99 105; 4 heads,
// width 512, 3 layers: 106 106 112 112, 90 103 110 122.
#define L_STEP_KEYS 4096
struct LatentStep {
    LatentShape w;
    const float *freq, *q;  // q[H hq]: the projected queries
    float *qa;              // [H][ld]: the queries on the cached rows
    const uint16_t *ukv;
    int ldu;
    const float *in, *kvnorm;  // the token's projected row
    float *cache, *part;       // part: H splits (L_STEP_RANK + 4) floats
    unsigned *count;           // [2 H], zero between launches
    float *out;
    int64_t cols;  // out up to which is zeroed behind the heads
    const DecodeCtl *ctl;
    int splits;
};
bool k_step_fits(const LatentShape &w, int ldu, const RowsArgs &uq, const RowsArgs &up, int up_pro, const RowsArgs &down, int down_pro,
                 int n_cu);
// uq: RP_NORM, the rows of the projected queries, then a.qa and the token's cache row from them; up: pro (RP_NORM or RP_UP), RE_GLU
hipError_t k_step_pair(hipStream_t s, const LatentStep &a, const RowsArgs &uq, const RowsArgs &up, int pro, int n_cu);
// down: pro (RP_PLAIN or RP_DOWN), RE_RESID; stride: from row to row of it (0: its ld)
hipError_t k_step_latent(hipStream_t s, const LatentStep &a, const RowsArgs &down, int64_t stride, int pro, int n_cu);
