// AddressSanitizer / UndefinedBehaviorSanitizer run of the library's host-only arithmetic: the plan, offsets and
// typed-piece tables of the streaming decode kernel (csrc/k_flow.hip, included as source; only its host functions run)
// and the synthetic-weight quantizers (csrc/synth.cpp).  No GPU call is made.  Every table entry is checked against the
// stream's bounds, which is what a wrong offset on the device would break.  Built and run by tests/test_sanitizers.py
// (hipcc with the sanitizers on the host side only).
#include "../../llama2.jl_amd/csrc/k_flow.hip"
#include "../../llama2.jl_amd/csrc/synth.cpp"
#include "../../llama2.jl_amd/csrc/delta_plan.h"
#include "../../llama2.jl_amd/csrc/draw.h"
#include "../../llama2.jl_amd/csrc/host_box.h"
#include "../../llama2.jl_amd/csrc/rows_plan.h"
#include "../../llama2.jl_amd/csrc/tiles_plan.h"

#include <stdio.h>

#include <string>
#include <vector>

static int fails = 0;
#define EXPECT(c)                                                 \
    do {                                                          \
        if (!(c)) {                                               \
            printf("line %d: %s\n", __LINE__, #c);                \
            fails++;                                              \
        }                                                         \
    } while (0)

static void check_shape(int dim, int hidden, int n_layers, int n_heads, int n_kv, int vocab, int seq_len, const int *layer7,
                        int cls_type, int kv16, bool expect_fit, bool cls_pairs = false) {
    const int grid = 256;
    FlowArgs a{};
    a.dim = dim, a.hidden = hidden, a.n_layers = n_layers, a.n_heads = n_heads, a.n_kv_heads = n_kv;
    a.hs = dim / n_heads, a.kv_dim = a.hs * n_kv, a.seq_len = seq_len, a.vocab = vocab, a.kv16 = kv16;
    std::vector<int> types;
    for (int l = 0; l < n_layers; l++)
        for (int k = 0; k < 7; k++) types.push_back(layer7[k]);
    std::string why;
    const bool fit = k_flow_plan(a, types.data(), (int)types.size(), cls_type, grid, &why, cls_pairs);
    EXPECT(fit == expect_fit);
    if (!fit) {
        EXPECT(!why.empty());
        return;
    }
    if (a.f32) return;  // no streams
    const FlowGeom g4[4] = {a.qkv, a.wo, a.w13, a.w2};
    for (int k = 0; k < 4; k++) {
        // every logical row has an owner, and the wavefronts' runs tile a workgroup's pieces exactly
        int64_t rows = 0;
        for (int wg = 0; wg < grid; wg++) {
            const int n = flow_n_local(g4[k], wg);
            rows += n;
            int pieces = 0;
            for (int w = 0; w < FLOW_NW; w++) {
                EXPECT(flow_wave_start(g4[k], wg, w) == pieces);
                pieces += flow_wave_pieces(g4[k], wg, w);
            }
            EXPECT(pieces == flow_wg_pieces(g4[k], wg));
            EXPECT(flow_half(g4[k]) ? pieces * 2 == n * flow_half(g4[k]) : pieces == n * g4[k].ppr);
            EXPECT(n <= FLOW_MAX_ROWS && pieces <= FLOW_MAX_PIECES / 4);
            if (flow_half(g4[k])) {
                // rows that end inside a piece: the pieces of a pair of rows hold every super-block of both rows once
                const int nb = 4 * flow_half(g4[k]);
                EXPECT(nb * 256 == dim && n % 2 == 0 && flow_half(g4[k]) % 2 == 1);
                std::vector<char> seen((size_t)n * nb, 0);
                for (int j = 0; j < pieces; j++) {
                    const int lr = flow_piece_row(g4[k], j), part = j % flow_half(g4[k]);
                    for (int b = 0; b < 8; b++) {
                        const int pb = 8 * part + b, odd = pb >= nb, blk = pb - odd * nb;
                        EXPECT(lr + odd < n && blk < nb);
                        EXPECT(!seen[(size_t)(lr + odd) * nb + blk]);
                        seen[(size_t)(lr + odd) * nb + blk] = 1;
                    }
                }
                for (char c : seen) EXPECT(c);
            }
        }
        EXPECT(rows == g4[k].n_rows);
    }
    if (a.mixed) {
        FlowTypedTables t;
        k_flow_typed_tables(a, types.data(), cls_type, grid, t);
        EXPECT(t.wave_off.size() == (size_t)grid * FLOW_NW && t.piece_off.size() == t.piece_tag.size());
        const int cls_piece = cls_type == L2H_TYPE_Q6_K ? FLOW_Q6_PIECE : FLOW_SLOT;
        for (size_t wi = 0; wi < t.wave_off.size(); wi++) {
            const int wg = (int)(wi / FLOW_NW), w = (int)(wi % FLOW_NW);
            const int64_t end = wi + 1 < t.wave_off.size() ? t.wave_off[wi + 1] : t.total - 4096;
            const int64_t first = t.piece_base[wi], last = wi + 1 < t.piece_base.size() ? t.piece_base[wi + 1] : (int64_t)t.piece_off.size();
            int64_t at = 0;
            for (int64_t e = first; e < last; e++) {
                const int ty = t.piece_tag[(size_t)e] & 0xFF;
                EXPECT(ty >= 0 && ty <= 2);
                EXPECT(t.piece_off[(size_t)e] == at);  // pieces lie back to back in consumption order
                at += flowm_piece_bytes(ty);
                // the tag names the type of the piece FLOWM_D places on (3: there is none)
                const int nxt = t.piece_tag[(size_t)e] >> 8;
                EXPECT(e + FLOWM_D < last ? nxt == (t.piece_tag[(size_t)(e + FLOWM_D)] & 0xFF) : nxt == 3);
            }
            EXPECT(t.cls_off[wi] == at);
            at += (int64_t)flow_wave_pieces(a.cls, wg, w) * cls_piece;
            EXPECT(t.wave_off[wi] + at <= end);
            EXPECT(t.wave_off[wi] % 256 == 0);
        }
    } else {
        std::vector<int64_t> off;
        const int64_t total = k_flow_offsets(a, cls_type, grid, off);
        EXPECT(off.size() == (size_t)grid * FLOW_NW);
        const int cls_piece = cls_type == L2H_TYPE_Q6_K ? FLOW_Q6_PIECE : FLOW_SLOT;
        for (size_t wi = 0; wi < off.size(); wi++) {
            const int wg = (int)(wi / FLOW_NW), w = (int)(wi % FLOW_NW);
            const int64_t end = wi + 1 < off.size() ? off[wi + 1] : total - 4096;
            const int64_t ring = (int64_t)n_layers * flow_layer_bytes(g4, wg, w, 4);
            const int64_t regs = (int64_t)n_layers * flow_layer_regs(g4, wg, w, 4) * FLOW_SLOT;
            EXPECT(flow_reg_base(g4, a.cls, cls_piece, n_layers, wg, w) == ring + (int64_t)flow_wave_pieces(a.cls, wg, w) * cls_piece);
            EXPECT(off[wi] + flow_reg_base(g4, a.cls, cls_piece, n_layers, wg, w) + regs <= end);
            EXPECT(off[wi] % 256 == 0);
        }
    }
    // logical row -> (tensor, row): a bijection onto the tensors' rows (both RoPE layouts, head sizes that are not powers of two)
    for (int neox = 0; neox < 2; neox++) {
        std::vector<char> seen((size_t)dim + 2 * a.kv_dim, 0);
        for (int L = 0; L < dim + 2 * a.kv_dim; L++) {
            int seg, row;
            flow_row_src(0, L, dim, a.kv_dim, a.hs, neox, seg, row, true);
            const int at = seg == 0 ? row : (seg == 1 ? dim + row : dim + a.kv_dim + row);
            EXPECT(seg >= 0 && seg <= 2 && row >= 0 && row < (seg == 0 ? dim : a.kv_dim));
            EXPECT(!seen[(size_t)at]);
            seen[(size_t)at] = 1;
        }
    }
}

// workgroups of the kernels for small models: 0 where the model does not go there
static int small(int type, int dim, int hidden, int heads, int kv, int vocab, int seq_len = 320, bool automatic = true) {
    FlowArgs a{};
    a.dim = dim, a.hidden = hidden, a.n_layers = 2, a.n_heads = heads, a.n_kv_heads = kv;
    a.hs = dim / heads, a.kv_dim = a.hs * kv, a.seq_len = seq_len, a.vocab = vocab;
    const std::vector<int> types(14, type);
    return k_flow_plan_small(a, types.data(), 14, type, 256, automatic);
}
static void check_small_plan() {
    // fp32, dim 256 or 512: hidden sizes at which a phase has pairs of rows for every workgroup, and wavefronts for every pair
    EXPECT(!small(0, 512, 44, 16, 16, 500) && small(0, 512, 48, 16, 16, 500) == 64 && small(0, 512, 3840, 16, 4, 500) == 256 && !small(0, 512, 3844, 16, 4, 500));
    EXPECT(small(0, 512, 244, 8, 8, 500) == 128 && small(0, 512, 248, 8, 8, 500) == 256 && small(0, 512, 3968, 8, 2, 500) == 256 && !small(0, 512, 3972, 8, 2, 500));
    EXPECT(!small(0, 512, 56, 4, 4, 500) && small(0, 512, 60, 4, 4, 500) == 64 && small(0, 512, 4032, 4, 1, 500) == 256 && !small(0, 512, 4036, 4, 4, 500));
    EXPECT(!small(0, 256, 52, 8, 8, 500) && small(0, 256, 56, 8, 8, 500) == 64 && small(0, 256, 1920, 8, 1, 500) == 128 && !small(0, 256, 1924, 8, 1, 500));
    EXPECT(small(0, 256, 1984, 4, 4, 500) == 128 && !small(0, 256, 1988, 4, 4, 500) && !small(0, 256, 688, 2, 2, 500) && !small(0, 1024, 2048, 16, 16, 500));
    // k-quants, dim 512 or 1024, heads of 32 or 64
    EXPECT(small(12, 512, 256, 8, 8, 65536) == 128 && !small(12, 512, 256, 8, 8, 65537) && small(12, 512, 3840, 8, 8, 500) == 128 && !small(12, 512, 4096, 8, 8, 500));
    EXPECT(small(13, 512, 3584, 16, 4, 500) == 128 && !small(13, 512, 3840, 16, 4, 500) && small(14, 1024, 3584, 32, 8, 500) == 256 && !small(14, 1024, 3840, 32, 8, 500));
    EXPECT(small(12, 1024, 3840, 16, 4, 131072) == 256 && !small(12, 1024, 3840, 16, 4, 131073) && !small(12, 1024, 4096, 16, 4, 500));
    EXPECT(!small(12, 1024, 1024, 8, 8, 500) && !small(12, 256, 512, 8, 8, 500) && !small(12, 512, 1024, 8, 2, 500, 320, false));
    // a long cache's attention wants at least half of the compute units
    EXPECT(small(0, 512, 64, 8, 8, 32000, 8192) == 64 && small(0, 512, 64, 8, 8, 32000, 8193) == 0);
    EXPECT(small(0, 512, 200, 8, 8, 32000, 8192) == 128 && small(0, 512, 200, 8, 8, 32000, 32768) == 128 && small(0, 512, 1376, 8, 8, 32000, 32768) == 256);
    EXPECT(small(0, 256, 64, 8, 8, 32000, 320) == 64 && small(0, 256, 64, 8, 8, 32000, 32768) == 0 && small(0, 256, 688, 8, 8, 32000, 32768) == 128);
}

// which kernel takes a product of a layered model: `each` positions for each of `experts` matrices (0: one matrix, `each` positions)
static bool few(int prec, int experts, int64_t cols, int each, int ld = 1024) {
    GemmTile tile{};
    GemmArgs a;
    a.n_rows = cols;
    a.ld = ld;
    a.matrices = experts;
    a.M = experts ? experts * each : each;
    a.rows_each = each;
    a.tiles = experts ? &tile : nullptr;
    return k_few_pays(a, prec, cols);
}
static void check_product_rule() {
    // bf16, sizes at which the one or the other takes at least 1.15 times as long (measured), and where the smaller kernel is up to 8 % behind
    EXPECT(few(0, 96, 4096, 48) && !few(0, 8, 512, 64) && few(0, 0, 32000, 128) && !few(0, 0, 32000, 160));
    // ... by the number of inputs, where the other takes 1.1 to 3.3 times as long
    EXPECT(!few(0, 0, 32000, 128, 512) && !few(0, 0, 16384, 128, 256) && few(0, 0, 8192, 128, 256) && few(0, 0, 32000, 64, 192));
    EXPECT(!few(0, 64, 4096, 60, 64) && !few(0, 16, 4096, 60, 256) && !few(0, 64, 1024, 60, 1024) && few(0, 16, 512, 60, 64) && few(0, 32, 512, 60, 512) && few(0, 32, 1024, 60, 2048));
    // plain ones against the library's, alone and with another launch behind it
    const uint16_t rows[1] = {};
    for (const uint16_t *emb : {(const uint16_t *)nullptr, rows}) {
        GemmArgs a;
        a.emb = emb;
        a.M = 333, a.n_rows = 256, a.ld = 4096;
        EXPECT(k_few_plain_pays(a) == (emb != nullptr));
        a.ld = 2048;
        EXPECT(k_few_plain_pays(a));
        a.M = 512, a.n_rows = 2048, a.ld = 256;
        EXPECT(k_few_plain_pays(a) == (emb != nullptr));
        a.n_rows = 4096;
        EXPECT(!k_few_plain_pays(a));
    }
    // fp32, 1.1 times: one matrix ...
    EXPECT(!few(1, 0, 1024, 509) && !few(1, 0, 4096, 64) && !few(1, 0, 512, 509) && !few(1, 0, 32000, 24) && !few(1, 0, 32000, 2048) && !few(1, 0, 8192, 160));
    EXPECT(!few(1, 0, 9216, 128) && !few(1, 0, 14336, 96) && !few(1, 0, 32000, 64) && !few(1, 0, 32000, 256));
    EXPECT(few(1, 0, 256, 509) && few(1, 0, 2048, 64) && few(1, 0, 4096, 17) && few(1, 0, 8192, 16) && few(1, 0, 128256, 1) && few(1, 0, 16, 2048));
    // ... and several
    EXPECT(!few(1, 16, 1024, 64) && !few(1, 16, 2048, 32) && !few(1, 64, 512, 48) && !few(1, 8, 64, 128) && !few(1, 32, 16, 100) && !few(1, 4, 64, 512));
    EXPECT(few(1, 8, 512, 32) && few(1, 16, 512, 16) && few(1, 8, 1024, 1) && few(1, 16, 256, 64) && few(1, 64, 32, 48));
}

// a decode product's workgroups have the LDS they need at every size that a model may have
static void check_rows_plan() {
    for (int n_cu : {32, 256})
        for (int K : {1, 700, 2048, 8192, 32768, 36864})
            for (int64_t rows : {(int64_t)1, (int64_t)255, (int64_t)32768, (int64_t)262144, (int64_t)1600000, (int64_t)20000000})
                for (int pro : {RP_PLAIN, RP_NORM, RP_UP, RP_DOWN})
                    for (int top : {1, 9, 64}) {
                        RowsArgs a;
                        a.K = K, a.ld = (K + 63) / 64 * 64, a.n_rows = rows, a.top = top, a.n_experts = 1024;
                        if (pro == RP_DOWN && (int64_t)top * a.ld > 36864) continue;
                        if (pro == RP_NORM && K > 32768) continue;
                        for (int u : {1, 2, 4}) {
                            const int64_t n = rows_grid(a, pro, n_cu, u), pairs = (rows + 1) / 2;
                            EXPECT(n >= 1 && n <= pairs && rows_lds(a, pro, pairs / n + 1) <= ROWS_LDS);
                        }
                    }
    // a grid made for two workgroups a CU has two there: the kernels' own LDS, as the compiler lays it out (96 bytes, 352 with a choice that is handed on, 2464
    // with one made), comes on top of the vectors and results, in whole units of 1280 bytes
    for (int pro : {RP_PLAIN, RP_NORM, RP_UP, RP_DOWN})
        for (int K = 18432; K <= 20480; K += 64)
            for (int64_t rows : {(int64_t)1024, (int64_t)40000, (int64_t)262144}) {
                RowsArgs a;
                a.K = a.ld = K, a.n_rows = rows, a.top = 1, a.n_experts = 8;
                const size_t own = pro == RP_UP ? 2464 : pro == RP_DOWN ? 352 : 224, lds = rows_lds(a, pro, (rows + 1) / 2 / 512 + 1) + own;
                if (rows_most(a, pro, 256) == 512) EXPECT(2 * ((lds + 1279) / 1280) * 1280 <= 160 * 1024);
            }
}

// quotients without a division, where rounding could show: around multiples, over all of the range
static void check_rows_div() {
    for (unsigned d = 1; d < 70000; d += d < 3000 ? 1 : 61) {
        const RowsDiv v = rows_div(d);
        for (unsigned long long k = 0; k * d < 0x80000000ull; k += 1 + k / 7)
            for (long long n : {(long long)(k * d) - 1, (long long)(k * d), (long long)(k * d + d / 2), 0x7FFFFFFFll})
                if (n >= 0 && n < 0x80000000ll) EXPECT(rows_quot((unsigned)n, v) == (unsigned)n / d);
    }
}

// the delta rule's scratch holds what every prompt of up to its length takes of it, and is not more than the outputs and records of chunks of 16 tokens
// by what the rule says; with less memory, fewer chunks a pass
static void check_delta_plan() {
    for (int D : {1, 64, 65, 128, 192, 256})
        for (int V : {1, 16, 100, 128, 129, 256})
            for (int H : {1, 8, 16, 32, 33, 100, 768})
                for (int cap : {256, 512, 768, 2048}) {
                    if (H * V > 32768) continue;
                    const DeltaShape d{H, 1, D, V, 4, 8, 8, 1e-5f};
                    const DeltaScratch s = delta_walk_scratch(d, cap);
                    const int64_t chunk = delta_chunk_floats(d);
                    EXPECT(s.least >= 1 && s.least <= s.floats && s.least <= std::max(chunk, delta_rec16_floats(d, cap)));
                    EXPECT(s.floats <= std::max(delta_rec16_floats(d, cap), std::max((int64_t)40 << 20, 8 * chunk)));
                    for (int64_t floats : {s.floats, s.least})
                        for (int M = L_DELTA_WALK_MIN; M <= cap; M++) {
                            if (!delta_wide_chunks(d, M)) {
                                EXPECT(delta_rec16_floats(d, M) <= floats && (M + 15) / 16 * 16 <= delta_out_rows(d, cap));
                                continue;
                            }
                            const int n = delta_pass_chunks(d, M, floats);
                            EXPECT(n >= 1 && n * chunk <= floats);
                        }
                    EXPECT(delta_out_rows(d, cap) >= L_DELTA_WALK_MIN - 1 && delta_out_rows(d, cap) <= cap);
                }
    // the most there is, 128 heads of 256 x 256, takes what chunks of 16 do; 16 of 128 x 128 are one pass, 48 three
    const DeltaShape many{128, 1, 256, 256, 4, 8, 8, 1e-5f}, few{16, 16, 128, 128, 4, 8, 8, 1e-5f}, more{48, 48, 128, 128, 4, 8, 8, 1e-5f};
    EXPECT(delta_walk_scratch(many, 2048).floats == delta_rec16_floats(many, 2048) && !delta_wide_chunks(many, 2048));
    EXPECT(delta_pass_chunks(few, 2048, delta_walk_scratch(few, 2048).floats) == 64 && delta_wide_chunks(few, 48));
    EXPECT(delta_pass_chunks(more, 2048, delta_walk_scratch(more, 2048).floats) == 22 && delta_wide_chunks(more, 48));
    for (int64_t room = 0; room <= 100; room++)
        for (int64_t have : {0, 3, 10, 50, 64, 80}) {
            int asked = 0;
            const int64_t n = delta_scratch_get(DeltaScratch{64, 5}, have, [&](int64_t k) {
                EXPECT(k > have && k >= 5 && k <= 64);
                asked++;
                return k <= room;
            });
            EXPECT(n == 0 ? have < 5 && room < 5 : n >= 5 && (n == have || (n <= room && 2 * n >= std::min<int64_t>(room, 64))));
            EXPECT(have < 64 || !asked);
        }
    // sizes at which the one or the other takes at least 1.05 times as long (measured)
    auto wide = [](int H, int D, int V, int M) { return delta_wide_chunks(DeltaShape{H, 1, D, V, 4, 8, 8, 1e-5f}, M); };
    EXPECT(wide(16, 64, 64, 2048) && wide(128, 64, 64, 2048) && wide(32, 128, 64, 2048) && wide(16, 128, 128, 2048) && wide(16, 256, 64, 2048) && wide(4, 256, 256, 2048) &&
           wide(8, 256, 256, 2048) && wide(16, 128, 256, 2048));
    EXPECT(!wide(128, 128, 128, 2048) && !wide(48, 192, 192, 2048) && !wide(16, 192, 192, 700) && !wide(64, 256, 256, 2048) && !wide(64, 128, 256, 2048) &&
           !wide(96, 64, 256, 2048) && !wide(32, 64, 256, 300) && !wide(8, 256, 256, 64) && !wide(32, 256, 128, 300));
}

// no step of the delta rule reads the slot of the ring that it writes
static void check_delta_ring() {
    for (int taps = 1; taps <= 64; taps++)
        for (int pos = 0; pos < 200; pos++)
            for (int j = 1; j < 70; j++) {
                const int slot = delta_ring_slot(taps, pos % taps, j);
                EXPECT(slot != pos % taps && slot < taps && (slot < 0 ? slot == -1 && j >= taps : j < taps));
                if (slot >= 0 && j <= pos) EXPECT(slot == (pos - j) % taps);
            }
}

// a context's pinned block and its models' boxes, with memory of the program's in place of pinned one: nothing is handed out twice, what does not fit
// is pinned by itself, what cannot be pinned is ordinary memory, and everything is given back (the sanitizer looks for leaks)
static int pins = 0;
static bool may_pin = true;
static void *test_pin(size_t bytes) {
    if (!may_pin) return nullptr;
    pins++;
    return malloc(bytes);
}
static void test_unpin(void *p) {
    pins--;
    free(p);
}
static void fill(HostBox &b, int64_t n, int with) {
    b.ctl[0].pos = b.ctl[1].pos = *b.pick = with;
    *b.gave_up = (unsigned)with;
    for (int64_t i = 0; i < n; i++) b.prompt[i] = b.out[i] = with;
}
static bool holds(const HostBox &b, int64_t n, int with) {
    bool ok = b.ctl[0].pos == with && b.ctl[1].pos == with && *b.pick == with && *b.gave_up == (unsigned)with;
    for (int64_t i = 0; i < n; i++) ok = ok && b.prompt[i] == with && b.out[i] == with;
    return ok;
}
static void check_boxes() {
    for (bool block : {true, false}) {
        may_pin = block;
        PinnedArena arena;
        arena.open(test_pin, test_unpin);
        EXPECT((arena.mem != nullptr) == block && pins == (int)block);
        const int64_t n[7] = {1, 500, 512, 4096, 20000, 1000, 40000};  // (the last takes more than the block)
        for (int round = 0; round < 3; round++) {
            may_pin = round != 1;
            std::vector<HostBox> boxes(35);
            for (size_t i = 0; i < boxes.size(); i++) {
                EXPECT(boxes[i].make(arena, n[i % 7]));
                fill(boxes[i], n[i % 7], (int)i + 1);
                // asked again, a model keeps what it has
                const void *mem = boxes[i].mem;
                std::vector<bool> used(arena.used, arena.used + PinnedArena::UNITS);
                EXPECT(boxes[i].make(arena, n[i % 7]) && boxes[i].mem == mem && std::equal(used.begin(), used.end(), arena.used) && holds(boxes[i], n[i % 7], (int)i + 1));
                if (i % 7 == 6) EXPECT(boxes[i].pinned == may_pin);
                EXPECT(boxes[i].seen == (boxes[i].pinned || (block && i % 7 != 6 && (const char *)boxes[i].mem >= arena.mem && (const char *)boxes[i].mem < arena.mem + PinnedArena::UNIT * PinnedArena::UNITS)));
            }
            for (size_t i = 0; i < boxes.size(); i++) EXPECT(holds(boxes[i], n[i % 7], (int)i + 1));
            // places in the middle that come free are used again
            if (block) {
                const void *at = boxes[1].mem;
                EXPECT((const char *)at >= arena.mem && (const char *)at < arena.mem + PinnedArena::UNIT * PinnedArena::UNITS);
                boxes[1].release(arena);
                EXPECT(!boxes[1].mem && boxes[1].make(arena, 500) && boxes[1].mem == at);
            }
            for (HostBox &b : boxes) b.release(arena);
            for (bool u : arena.used) EXPECT(!u);
            EXPECT(pins == (int)block);
        }
        arena.close();
        EXPECT(pins == 0);
    }
}

// every tile of a prompt's product is taken exactly once, as a whole or as both of its halves
static void check_tiles_plan() {
    for (int n_cu : {32, 64, 250, 256}) {
        int split = 0;
        for (unsigned n = 1; n <= 2048; n++)
            for (int halves = 0; halves < 2; halves++) {
                const TilesPlan p = tiles_plan(n, halves != 0, n_cu);
                std::vector<int> taken(n, 0);  // in halves
                const unsigned grid = tiles_grid(p);
                for (unsigned b = 0; b < grid; b++) {
                    const TilesWork w = tiles_work(p, b);
                    if (!w.any) continue;
                    EXPECT(w.item < n && w.half >= -1 && w.half <= 1);
                    if (w.item >= n) continue;
                    EXPECT((taken[w.item] & (w.half < 0 ? 3 : 1 << w.half)) == 0);
                    taken[w.item] |= w.half < 0 ? 3 : 1 << w.half;
                }
                bool all = true;
                for (unsigned i = 0; i < n; i++) all = all && taken[i] == 3;
                if (!all) printf("%u tiles\n", n);
                EXPECT(all);
                // whole rounds, and no more than one round of halves behind them
                EXPECT(p.whole == n || (halves && p.whole % (unsigned)n_cu == 0 && 2 * (n - p.whole) <= (unsigned)n_cu));
                split += p.whole < n;
            }
        EXPECT(n_cu != 256 || split == 7 * 128);
    }
    // an expert's blocks have all of its units once, in shares that differ by one at most and are within the bound; all blocks fit the lists and grids
    for (unsigned b = 1; b <= TILES_MAX_UNITS; b++) {
        for (unsigned units = 0; units <= 400; units++) {
            const TilesSplit v = tiles_split(units, b);
            EXPECT(v.blocks == (units + b - 1) / b && v.largest <= b);
            unsigned at = 0, weight = 0;
            const TilesShares share(units, v.blocks);
            for (unsigned k = 0; k < v.blocks; k++) {
                const unsigned u = share.at(k + 1) - at;
                EXPECT(share.at(k) == at && u >= 1 && u <= v.largest && u + 1 >= v.largest);
                at += u;
                weight += tiles_weight(u);
            }
            EXPECT(at == units && weight == v.weight);
        }
        unsigned seed = 7 * b;
        for (int experts : {1, 2, 7, 64, 300}) {
            int64_t rows = 0, blocks = 0;
            for (int e = 0; e < experts; e++) {
                seed = seed * 1664525u + 1013904223u;
                const int64_t n = e % 3 == 0 ? 1 : (seed >> 20) % 700;
                rows += n;
                blocks += tiles_split((unsigned)((n + TILES_UNIT - 1) / TILES_UNIT), b).blocks;
            }
            EXPECT(blocks <= tiles_most(rows, experts, b) && tiles_most(rows, experts, b) <= tiles_most(rows, experts, 1));
        }
    }
    // what the rule was made from: the bound of the least time at each (rows, experts, row groups, steps)
    EXPECT(tiles_bound(8192, 32, 4, 32, 256) == 3 && tiles_bound(8192, 32, 8, 16, 256) == 5 && tiles_bound(8192, 32, 16, 64, 256) == 5);
    EXPECT(tiles_bound(1332, 16, 8, 64, 256) == 1 && tiles_bound(1332, 16, 16, 32, 256) == 2 && tiles_bound(8000, 16, 8, 32, 256) == 5);
    // where few experts have most rows: what the launch that counts them chooses, and the lists and grids it has for that
    auto units_of = [](const TilesRule &r, const std::vector<int> &rows) {
        unsigned n[2] = {0, 0}, weight[2] = {0, 0};
        for (int v : rows)
            for (int w = 0; w < 2; w++) {
                const TilesSplit k = tiles_split((unsigned)(v + TILES_UNIT - 1) / TILES_UNIT, w ? TILES_WHOLE_UNITS : r.bound);
                n[w] += k.blocks, weight[w] += k.weight;
            }
        const bool whole = r.n_cu && tiles_rounds(r, n[1], weight[1]) < tiles_rounds(r, n[0], weight[0]);
        int64_t total = 0;
        for (int v : rows) total += v;
        EXPECT(n[whole] <= tiles_most(total, (int)rows.size(), r) && tiles_most(total, (int)rows.size(), r) <= tiles_most(total, (int)rows.size(), 1));
        return whole ? TILES_WHOLE_UNITS : (int)r.bound;
    };
    auto crowd = [](int experts, int n, int m) {  // n of them have m rows each, the others a share of what is left of 4 m
        std::vector<int> rows(experts, (4 - n) * m / (experts - n));
        for (int e = 0; e < n; e++) rows[e] = m;
        return rows;
    };
    // (experts, crowded ones, positions, row groups, steps: blocks of whole tiles are faster by 5 to 24 %, and the bound by 15 to 40 %)
    EXPECT(units_of(tiles_rule(2000, 16, 14, 56, 256), crowd(16, 2, 500)) == 4 && units_of(tiles_rule(8000, 16, 8, 32, 256), crowd(16, 4, 2000)) == 4);
    EXPECT(units_of(tiles_rule(8000, 16, 16, 64, 256), crowd(16, 1, 2000)) == 4 && units_of(tiles_rule(8000, 32, 8, 32, 256), crowd(32, 2, 2000)) == 4);
    EXPECT(units_of(tiles_rule(4000, 16, 8, 32, 256), crowd(16, 4, 1000)) == 3 && units_of(tiles_rule(2000, 16, 16, 64, 256), crowd(16, 4, 500)) == 3);
    EXPECT(units_of(tiles_rule(8192, 32, 16, 64, 256), std::vector<int>(32, 256)) == tiles_rule(8192, 32, 16, 64, 256).bound);
    for (int experts : {1, 2, 5, 16, 70, 1000})
        for (int m : {1, 63, 700, 4096, 100000})
            for (unsigned n_nt : {1u, 16u, 200u})
                for (int n = 0; n <= std::min(experts - 1, 4); n++) {
                    const std::vector<int> rows = crowd(experts, n, m);
                    int64_t total = 0;
                    for (int v : rows) total += v;
                    if (total) units_of(tiles_rule(total, experts, n_nt, 64, 256), rows);
                }
    // a grouped product's grid is made for the most tiles there can be, and dealt out by how many there are
    for (unsigned most = 1; most <= 300; most++)
        for (unsigned n = 1; n <= most; n++) {
            std::vector<int> taken(n, 0);
            for (unsigned b = 0; b < tiles_workgroups(most); b++) {
                const unsigned i = tiles_deal(n, b);
                if (i < n) taken[i]++;
            }
            for (int t : taken) EXPECT(t == 1);
        }
}

// a draw's running sums as a workgroup of the draw kernels forms them: in wavefronts by doubling distances, then wavefront by wavefront
struct DrawSums {
    std::vector<double> own, lower, end;
    double all = 0.0;
    explicit DrawSums(const std::vector<double> &v) : own(v), lower(v.size()), end(v.size()) {
        for (size_t w0 = 0; w0 < v.size(); w0 += 64) {
            double x[64], y[64];
            for (int l = 0; l < 64; l++) x[l] = v[w0 + l];
            for (int d = 1; d < 64; d *= 2) {
                for (int l = 0; l < 64; l++) y[l] = x[l] + (l >= d ? x[l - d] : 0.0);
                for (int l = 0; l < 64; l++) x[l] = y[l];
            }
            for (int l = 0; l < 64; l++) {
                lower[w0 + l] = all + (l ? x[l - 1] : 0.0);
                end[w0 + l] = all + x[l];
            }
            all += x[63];
        }
    }
    int owner(double target) const {
        int first = -1, last = -1;
        for (int t = 0; t < (int)own.size(); t++) {
            if (own[t] > 0.0) last = t;
            if (first < 0 && draw_reaches(own[t], end[t], target)) first = t;
        }
        return first < 0 ? last : first;
    }
};
// Every target has an owner and a pick that has weight: at every border between two threads and the numbers beside it, with probabilities of the same size,
// of very different sizes and many of zero.  The pick is where the running sum in order reaches the target, within what two orders of the sum can differ by.
static void check_draw() {
    unsigned long long seed = 12345;
    auto uniform = [&] { return (double)((seed = seed * 6364136223846793005ull + 1442695040888963407ull) >> 40) / 16777216.0; };
    for (int round = 0; round < 24; round++) {
        const int n = round % 3 == 0 ? 4096 : round % 3 == 1 ? 8 : 1000 + (int)(3000 * uniform());
        std::vector<float> p(n);
        double sum = 0.0;
        for (float &v : p) {
            const double z = round % 4 == 0 ? 6 * uniform() : round % 4 == 1 ? 60 * uniform() : uniform() < 0.6 ? 200.0 : 20 * uniform();
            v = (float)exp(-z);
            sum += (double)v;
        }
        if (round == 1) {  // logits -37.82 four times, 0, -200 three times
            for (int i = 0; i < 8; i++) p[i] = i < 4 ? (float)exp(-37.82) : i == 4 ? 1.0f : 0.0f;
            sum = 1.0;
        }
        for (float &v : p) v /= (float)sum;
        std::vector<double> own(1024, 0.0), cum(n + 1, 0.0);
        for (int i = 0; i < n; i++) {
            own[i / 4] += (double)p[i];
            cum[i + 1] = cum[i] + (double)p[i];
        }
        const DrawSums s(own);
        for (int t = 0; t + 1 < 1024; t++) EXPECT(s.end[t] == s.lower[t + 1]);
        const double slack = 1024 * 2.3e-16 * s.all;
        for (int t = 0; 4 * t < n; t++)
            for (int k = 0; k < 8; k++) {
                // (below and above the thread's two ends, what the difference of its end and its own sum comes to, and a number inside)
                const double at = k < 3 ? s.end[t] : k < 6 ? s.end[t] - own[t] : s.lower[t] + uniform() * own[t];
                const double target = k % 3 == 1 ? nextafter(at, 0.0) : k % 3 == 2 ? nextafter(at, 2.0) : at;
                if (!(target > 0.0 && target <= s.all)) continue;
                const int owner = s.owner(target);
                EXPECT(owner >= 0 && 4 * owner < n);
                if (owner < 0 || 4 * owner >= n) return;
                DrawWalk walk(s.lower[owner], target);
                for (int i = 4 * owner; i < std::min(n, 4 * owner + 4); i++) walk.next(i, p[i]);
                EXPECT(p[walk.pick] > 0.0f && cum[walk.pick] <= target + slack && cum[walk.pick + 1] >= target - slack);
            }
    }
    // the example: the target lies above the end of the first four and far below the rest
    std::vector<double> v(1024, 0.0);
    for (int i = 0; i < 4; i++) v[0] += (double)(float)exp(-37.82);
    v[1] = 1.0;
    const DrawSums s(v);
    EXPECT(s.owner((double)2e-16f * s.all) == 1 && s.owner(1.5e-16) == 0);
}

int main() {
    check_draw();
    check_tiles_plan();
    check_small_plan();
    check_product_rule();
    check_rows_plan();
    check_rows_div();
    check_delta_plan();
    check_delta_ring();
    check_boxes();
    const int q4[7] = {12, 12, 12, 12, 12, 12, 12}, q5m[7] = {13, 13, 13, 13, 13, 14, 13}, mix[7] = {12, 12, 13, 12, 12, 14, 12},
              f32[7] = {0, 0, 0, 0, 0, 0, 0}, bad[7] = {12, 12, 12, 12, 12, 12, 13};
    check_shape(4096, 14336, 32, 32, 8, 128256, 512, q4, 14, 0, true);    // the headline model
    check_shape(4096, 14336, 32, 32, 8, 128256, 4096, q5m, 14, 0, true);  // q5_K_M mix: typed pieces
    check_shape(4096, 14336, 4, 32, 8, 128256, 512, mix, 12, 0, true);    // q4_K classifier behind typed pieces
    check_shape(3072, 8192, 32, 32, 32, 32064, 4096, q4, 12, 0, true);    // Phi-3: a piece and a half per row, head size 96
    check_shape(3072, 8192, 2, 32, 32, 32064, 4096, q4, 12, 1, true);     // the same with an fp16 cache
    check_shape(2048, 4096, 3, 16, 4, 1000, 160, q4, 14, 0, false);       // q6_K classifier needs 4096
    check_shape(2048, 4096, 3, 16, 4, 1000, 160, q4, 12, 0, true);
    check_shape(2048, 8192, 3, 16, 4, 1001, 160, q4, 14, 0, true, true);  // ... unless its rows may go in pairs
    check_shape(1792, 4096, 2, 28, 4, 999, 160, q5m, 14, 0, false, true); // (28 heads do not divide the workgroups)
    check_shape(1536, 4096, 2, 16, 4, 999, 160, mix, 14, 0, true, true);
    check_shape(1536, 2048, 2, 16, 16, 999, 96, q4, 12, 0, true);         // a quarter below 2048: padded rows
    check_shape(3072, 8192, 2, 32, 8, 32064, 512, mix, 12, 0, true);      // halves with typed pieces and grouped heads
    check_shape(1024, 2048, 2, 16, 16, 999, 96, q4, 12, 0, false);        // half below: refused
    check_shape(512, 1376, 8, 8, 8, 32000, 1024, f32, 0, 0, true);        // llama2.c shape
    check_shape(4096, 14336, 2, 32, 8, 32000, 512, bad, 14, 0, false);    // w1 and w3 of different types
    check_shape(4096, 14336, 2, 32, 8, 32000, 40000, q4, 14, 0, false);   // cache too long for the attention area
    // synthetic weights: every quantizer over a few thousand values, odd thread counts
    std::vector<float> x(256 * 37);
    for (int t = 1; t <= 5; t += 2) {
        EXPECT(l2h_synth_normal(7, 3, 11, (int64_t)x.size(), 0.02f, x.data(), t) == 0);
        for (int type : {12, 13, 14}) {
            const int64_t bb = type == 12 ? 144 : (type == 13 ? 176 : 210);
            std::vector<uint8_t> out((size_t)(x.size() / 256) * (size_t)bb);
            EXPECT(l2h_quantize_weights(type, x.data(), (int64_t)x.size(), out.data(), t) == 0);
        }
    }
    EXPECT(l2h_quantize_weights(12, x.data(), 100, x.data(), 1) != 0);
    if (fails) {
        printf("%d checks failed\n", fails);
        return 1;
    }
    puts("host arithmetic: sanitizers silent, tables consistent");
    return 0;
}
