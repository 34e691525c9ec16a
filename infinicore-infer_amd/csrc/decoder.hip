// The step function in native code: every kernel of a step issued by one call (host code only; the
// kernels are the library's own entry points).  The reference's is src/models/jiuge/jiuge.cpp:114-298.
//
// What runs for a layer depends on the step alone, never on the model, but for the decode steps of up to 8 rows that one kernel takes with all their layers
// (decode_chain.hip, for the sizes that it is built for).  Up to 16 rows in bfloat16 take the
// few-row products with their epilogues (rotary and cache write after QKV; residual add, the next norm's
// weight and sums of squares after O and down; SwiGLU after gate/up), the norm between two products being
// split over them; more rows take the products in tiles (QKV with rotary and cache write, gate/up with SwiGLU in
// the epilogue) or the library's, float32 the product of bfloat16 parts or the library's, as ic_product chooses, and the norm, rotary and activation kernels.
// Single-token rows go to the split-key attention kernel, prompt portions to the tiled one, both of a mixed step to one launch
// where that is faster, what neither takes to the general one.
#include "common.h"
#include "decode_chain.h"
#include "infinicore_infer_engine.h"
#include "infinicore_infer_variants.h"
#include <algorithm>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

namespace {

// The thresholds below are read by the ic_rule_* functions alone; the step function here and the parts' Python
// forward both ask those functions, so a rule is written once.
constexpr int kFewRows = 16;        // up to here the few-row products beat the library
constexpr int kMidRows = 64;        // up to here the sliced product beats it for results as wide as the model
// Layers from which on a decode step runs them in one launch.  Not a line of speed: each layer saves 6 us at one row of the 1B and 2B shapes (1B shape, 600 keys: 93.4 -> 79.8
// us with three layers, 223.8 -> 183.8 with eight), starting costs 4, so one and two layers would save 3 and 8 us too.  They stay kernel by kernel for the sake of
// comparison: such steps equal those issued from Python bit for bit, on the layer sizes that deeper models have.
constexpr int kChainMinEntries = 3;
constexpr int kMaxSumsqParts = 256; // column blocks of sums of squares a product takes as row factors

thread_local std::string g_create_error;

inline size_t align_up(size_t n, size_t a) { return (n + a - 1) / a * a; }
inline int dtype_size(int dtype) { return dtype == IC_BF16 ? 2 : 4; }

struct Workspace {
    // byte offsets into the caller's workspace
    size_t residual, normed, qkv, attn_out, mixer_out, ffn_out, mixer_tail, mixer_sumsq, ffn_tail, ffn_sumsq, gate_up, act,
        part_acc, part_ml, decode_order, head_in, tail_parts, tile_parts, f32_parts, chain, total;
};

// Rows whose norm is half done: values = x * w, sums of squares per column block; the row factor
// rsqrt(sum / width + eps) is applied by the product that consumes them.
struct Deferred {
    const void* values = nullptr;
    const float* sumsq = nullptr;
    int parts = 0, width = 0;
    float eps = 0.f;
};

}  // namespace

// ---- which kernel takes what: the one home of the dispatch rules ----------------------------------------------------------
IC_EXPORT int ic_rule_few_rows() { return kFewRows; }
IC_EXPORT int ic_rule_sumsq_parts_max() { return kMaxSumsqParts; }

IC_EXPORT int ic_rule_own_product(int a_dtype, int w_dtype, int c_dtype, int rows) {
    return rows <= kFewRows && a_dtype == IC_BF16 && ic_gemm_nt_supported(a_dtype, w_dtype, c_dtype);
}

IC_EXPORT int ic_rule_qkv_fused(int dtype, int rows, int K, int lda, int ldw, int head_dim, int rot_dim, int kv_heads_written,
                                int row_factors_owed) {
    if (dtype != IC_BF16 || kv_heads_written <= 0 || rot_dim != head_dim || !ic_gemm_qkv_rope_supported(IC_BF16, head_dim)) return 0;
    if (rows <= kFewRows) return 1;
    return !row_factors_owed && rows <= ic_gemm_nt_epilogue_rows(2, K, lda, ldw);
}

IC_EXPORT int ic_rule_qkv_tiles(int dtype, const void* A, const void* W, const void* C, int rows, int K, int lda, int ldw, int ldc, const float* cos_t,
                                const float* sin_t, const void* kcache, const void* vcache, int nh, int kv_heads_written, int head_dim, int rot_dim,
                                int page_size) {
    return dtype == IC_BF16 && kv_heads_written > 0 && rot_dim == head_dim &&
           ic_gemm_tiles_rope_supported(A, W, C, rows, K, lda, ldw, ldc, cos_t, sin_t, kcache, vcache, nh, kv_heads_written, head_dim, page_size) &&
           ic_gemm_tiles_pays(rows, (nh + 2 * kv_heads_written) * head_dim, K, 2);
}

IC_EXPORT int ic_rule_gate_up_fused(int dtype, int rows, int K, int lda, int ldw, int row_factors_owed) {
    if (dtype != IC_BF16) return 0;
    if (rows <= kFewRows) return 1;
    return !row_factors_owed && rows <= ic_gemm_nt_epilogue_rows(1, K, lda, ldw);
}

IC_EXPORT int ic_rule_gate_up_tiles(int dtype, const void* A, const void* W, const void* C, int rows, int N, int K, int lda, int ldw, int ldc) {
    const bool aligned = !(((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15);
    return dtype == IC_BF16 && aligned && ic_gemm_tiles_supported(rows, N, K, lda, ldw, ldc, 1) && ic_gemm_tiles_pays(rows, N, K, 1);
}

IC_EXPORT int ic_rule_tail(int dtype, int rows, int N, int K, int lda, int ldw) {
    if (dtype != IC_BF16 || rows <= 0) return IC_TAIL_PLAIN;
    if (rows <= kMidRows && N % 4 == 0 && ic_gemm_splitk_supported(rows, N, K, lda, ldw) && ic_gemm_splitk_pays(rows, N, K))
        return IC_TAIL_SLICES;
    if (rows <= kFewRows && ic_gemm_nt_residual_parts(N) <= kMaxSumsqParts) return IC_TAIL_SPLIT_NORM;
    return IC_TAIL_PLAIN;
}

IC_EXPORT int ic_rule_attention(int dtype, int head_dim, int page_size, int n_decode_rows, int n_tiles) {
    const bool dec_ok = ic_attn_decode_supported(dtype, head_dim) != 0;
    const bool pre_ok = ic_attn_prefill_supported(dtype, head_dim, page_size) != 0;
    const bool use_dec = dec_ok && n_decode_rows > 0 && (pre_ok || n_tiles == 0);
    const bool use_pre = pre_ok && n_tiles > 0 && (dec_ok || n_decode_rows == 0);
    if (!((use_dec || n_decode_rows == 0) && (use_pre || n_tiles == 0))) return IC_ATTN_GENERAL;
    return (use_dec ? IC_ATTN_SINGLE_TOKENS : 0) | (use_pre ? IC_ATTN_PORTIONS : 0);
}

// Together the two kinds of block fill each other's tails: 40 rows of 100..2,048 keys beside portions of 512 and 463 after 512 (24:8 heads of 64) 39.1 -> 25.2
// us, 8 rows beside a prompt of 300 18.2 -> 11.0 (36 heads of 64: 20.8 -> 14.6; 32:2 of 128: 23.9 -> 16.5), 60 rows of up to 3,000 keys beside 850
// tokens 44.2 -> 32.0 (87.6 -> 82.1, 45.1 -> 38.9).  Not where few tiles with long walks would take two wave groups each, which the common kernel does
// not have: 2 rows beside a portion of 700 after 2,500 (32:2 of 128) 71.2 -> 77.2.
IC_EXPORT int ic_rule_attention_together(int dtype, int nh, int nkvh, int head_dim, int page_size, int table_stride, int n_decode_rows, int n_tiles,
                                         int max_tile_position, int window, int parts, int compute_units) {
    if (n_decode_rows <= 0 || n_tiles <= 0 || !ic_attn_mixed_supported(dtype, nh, nkvh, head_dim, page_size, table_stride)) return 0;
    const int keys = window > 0 ? std::min(max_tile_position + 1, window + ic_attn_prefill_tile_rows()) : max_tile_position + 1;
    const bool two_groups = parts <= 1 && (long long)n_tiles * nh <= 2LL * (compute_units > 0 ? compute_units : 256);
    return !(two_groups && keys >= 24 * 64);
}

IC_EXPORT int ic_rule_context_bucket(int n_keys) {
    int b = 256;
    while (b < n_keys) b *= 2;
    if (b <= 1024) return b;
    const int q = b / 8;
    return (n_keys + q - 1) / q * q;
}

struct IcDecoder {
    IcDecoderMeta meta;
    std::vector<IcLayer> layers;
    std::vector<IcRunEntry> entries;
    int max_qkv_width = 0, max_attn_width = 0, max_intermediate = 0;
    std::vector<ChainEntry> table;       // of layers that are alike enough for one launch, else empty
    const ChainEntry* device_table = nullptr;      // the same on the device: steps may run the layers in one launch
    int* gave_up = nullptr;              // the caller's, see ic_decoder_use_layer_table
    std::string error;

    int fail(int status, const char* what, int entry) {
        char buf[256];
        if (entry >= 0) snprintf(buf, sizeof buf, "run-order entry %d (layer %d): %s returned %d", entry, entries[entry].layer, what, status);
        else snprintf(buf, sizeof buf, "%s returned %d", what, status);
        error = buf;
        return status;
    }

    // the last question put to ic_attn_decode_splits and its answer: the layers of a model mostly ask the same one
    mutable int split_key[7] = {-1, -1, -1, -1, -1, -1, -1}, split_answer = 1;

    int splits_for(const IcStepBatch& b, const IcAttention& a) const {
        if (b.fixed_decode_splits > 0) return b.fixed_decode_splits;
        const int matrix_cores = ic_attn_decode_on_matrix_cores(meta.dtype, a.n_heads, a.n_kv_heads);
        const int key[7] = {b.n_decode_rows, a.n_heads, a.n_kv_heads, a.head_dim, a.window, b.max_context, matrix_cores};
        if (memcmp(key, split_key, sizeof key) != 0) {
            split_answer = ic_attn_decode_splits(b.n_decode_rows, a.n_heads, a.n_kv_heads, a.head_dim, dtype_size(meta.dtype), a.window,
                                                 b.max_context, matrix_cores, meta.compute_units);
            memcpy(split_key, key, sizeof key);
        }
        return split_answer;
    }

    // The largest position of the prompt portions: a long chat that brings one token does not lengthen the tiles' walks.  With the whole step's in its
    // place parts are too long and too few: 16 chats of 1,073..8,000 keys beside 512 tokens after 2,000 (24:8 heads of 64) 41.6 -> 62.8 us, 12 of up to
    // 3,000 beside 500 after 400 27.6 -> 31.4; and steps that run best in one launch do not (32:2 of 128, 8 of up to 9,000 beside 700 and 90: 33.1 -> 40.6).
    // It costs up to 3 % where walks of 40 key tiles of 128 do better in two parts than in four (16 chats of up to 8,000 beside 512 after 2,000: 170 -> 175).
    static int tiles_end(const IcStepBatch& b) { return b.max_tile_position > 0 ? b.max_tile_position : b.max_position; }
    // into how many parts the walks of a step's prompt tiles are cut (1: not at all), and key tiles per part
    int tile_parts_for(const IcStepBatch& b, const IcAttention& a, int* part_len) const {
        if (!meta.attention_counters) { if (part_len) *part_len = 0; return 1; }     // no counters: no cut
        return ic_attn_prefill_parts_of_step(meta.dtype, b.n_prefill_tiles, a.n_heads, a.head_dim, tiles_end(b), a.window, meta.compute_units, part_len);
    }
    // the same where they run beside the step's single tokens
    int mixed_parts_for(const IcStepBatch& b, const IcAttention& a, int* part_len) const {
        if (!meta.attention_counters) { if (part_len) *part_len = 0; return 1; }
        return ic_attn_mixed_parts_of_step(meta.dtype, b.n_prefill_tiles, a.n_heads, a.head_dim, tiles_end(b), a.window, meta.compute_units, part_len);
    }

    ChainShape chain_shape() const {
        const IcLayer& l = layers[entries[0].layer];
        return ChainShape{meta.hidden, l.attention.n_heads, l.attention.n_kv_heads, l.attention.head_dim, l.ffn.intermediate, meta.page_size, meta.compute_units};
    }

    // All layers in one launch: every row a request's single new token, all logits wanted, memory in which its 16-byte accesses are aligned.
    bool takes_chain(const IcStepBatch& b, const void* workspace) const {
        return device_table && !((uintptr_t)workspace & 15) && b.fixed_decode_splits <= 0 && b.decode_rows_identity && b.want_rows_identity && b.n_want == b.n_tokens && b.n_decode_rows == b.n_tokens &&
               b.n_prefill_tiles == 0 && b.n_tokens <= kChainMaxRows && chain_supported(chain_shape(), b.n_tokens, meta.n_entries, std::max(b.max_context, b.max_position + 1));
    }

    // The layers' table, if they are alike enough for one launch.  Only what the description says: nothing is asked of the device, which other threads may be recording on.
    void make_table() {
        if (meta.dtype != IC_BF16 || meta.n_entries < kChainMinEntries) return;
        const IcRunEntry& e0 = entries[0];
        const IcLayer& l0 = layers[e0.layer];
        const IcAttention& a0 = l0.attention;
        if (a0.window != 0 || a0.shared_kv || a0.rot_dim != a0.head_dim || (((uintptr_t)a0.cos | (uintptr_t)a0.sin) & 15)) return;      // (such tables ic_gemm_qkv_rope refuses)
        std::vector<ChainEntry> made;
        for (const IcRunEntry& e : entries) {
            const IcLayer& l = layers[e.layer];
            const IcAttention& a = l.attention;
            if (!e.writes_cache || e.group != e0.group || a.n_heads != a0.n_heads || a.n_kv_heads != a0.n_kv_heads || a.head_dim != a0.head_dim || a.window != 0 ||
                a.shared_kv || a.rot_dim != a0.rot_dim || a.max_positions != a0.max_positions || a.softmax_scale != a0.softmax_scale || a.cos != a0.cos ||
                a.sin != a0.sin || l.mixer_norm.eps != l0.mixer_norm.eps || l.ffn_norm.eps != l0.ffn_norm.eps || l.ffn.intermediate != l0.ffn.intermediate ||
                l.residual_scale != l0.residual_scale) return;
            if (((uintptr_t)a.w_qkv | (uintptr_t)a.w_o | (uintptr_t)l.ffn.w_gate_up | (uintptr_t)l.ffn.w_down | (uintptr_t)e.k_cache | (uintptr_t)e.v_cache) & 15) return;
            for (const ChainEntry& other : made)
                if (other.k_cache == e.k_cache || other.v_cache == e.v_cache) return;
            made.push_back(ChainEntry{a.w_qkv, a.w_o, l.ffn.w_gate_up, l.ffn.w_down, l.mixer_norm.weight, l.ffn_norm.weight, e.k_cache, e.v_cache});
        }
        if (!chain_supported(chain_shape(), 1, meta.n_entries, 1)) return;
        ChainEntry end{};
        end.norm_in = meta.final_norm_scaled;
        made.push_back(end);
        table = std::move(made);
    }

    Workspace layout(const IcStepBatch& b) const {
        const size_t T = (size_t)b.n_tokens, d = (size_t)meta.hidden, ds = (size_t)dtype_size(meta.dtype);
        const int parts = ic_gemm_nt_residual_parts(meta.hidden);
        Workspace w{};
        size_t o = 0;
        auto take = [&](size_t bytes) { const size_t at = o; o = align_up(o + bytes, 256); return at; };
        w.residual = take(T * d * 4);
        w.normed = take(T * d * ds);
        w.qkv = take(T * (size_t)max_qkv_width * ds);
        w.attn_out = take(T * (size_t)max_attn_width * ds);
        w.mixer_out = take(T * d * ds);
        w.ffn_out = take(T * d * ds);
        const size_t few = std::min<size_t>(T, (size_t)ic_rule_few_rows());
        w.mixer_tail = take(few * d * 2);
        w.mixer_sumsq = take((size_t)parts * 16 * 4);
        w.ffn_tail = take(few * d * 2);
        w.ffn_sumsq = take((size_t)(device_table ? std::max(parts, chain_sumsq_parts(chain_shape())) : parts) * 16 * 4);
        w.gate_up = take(T * 2 * (size_t)max_intermediate * ds);
        w.act = take(T * (size_t)max_intermediate * ds);
        size_t acc = 0, ml = 0;      // partial results of the key splits: [row, head, split, head size] and [row, head, split, 2]
        if (b.n_decode_rows > 0)
            for (const IcLayer& l : layers) {
                const size_t cells = (size_t)b.n_decode_rows * l.attention.n_heads * (size_t)splits_for(b, l.attention);
                acc = std::max(acc, cells * l.attention.head_dim);
                ml = std::max(ml, cells * 2);
            }
        w.part_acc = take(acc * 4);
        w.part_ml = take(ml * 4);
        w.decode_order = take(b.decode_rows_identity ? (size_t)b.n_decode_rows * 4 : 0);
        w.head_in = take((size_t)b.n_want * d * ds);
        size_t slices = 0;           // the O and down products as slices over K, where that pays
        for (const IcLayer& l : layers)
            for (const int K : {l.attention.n_heads * l.attention.head_dim, l.ffn.intermediate})
                if (ic_rule_tail(meta.dtype, (int)T, meta.hidden, K, K, K) == IC_TAIL_SLICES)
                    slices = std::max(slices, (size_t)ic_gemm_splitk_slices(meta.hidden, K));
        w.tail_parts = take(slices * T * d * 4);
        size_t cut = 0;              // the states of prompt tiles whose walk over the keys is cut into parts
        if (meta.dtype == IC_BF16 && b.n_prefill_tiles > 0)
            for (const IcLayer& l : layers) {
                int len = 0;
                const int p = std::max(tile_parts_for(b, l.attention, &len), b.n_decode_rows > 0 ? mixed_parts_for(b, l.attention, &len) : 1);
                cut = std::max(cut, (size_t)ic_attn_prefill_scratch_floats(b.n_prefill_tiles, l.attention.n_heads, l.attention.head_dim, p));
            }
        w.tile_parts = take(cut * 4);
        long long f32 = 0;           // float32 products of many rows (this engine's own: another's must not write there between two launches)
        if (meta.dtype == IC_F32) {
            for (const IcLayer& l : layers) {
                const int heads = l.attention.n_heads * l.attention.head_dim, di = l.ffn.intermediate;
                f32 = std::max({f32, ic_gemm_f32_workspace_bytes(b.n_tokens, max_qkv_width, meta.hidden), ic_gemm_f32_workspace_bytes(b.n_tokens, meta.hidden, heads),
                                ic_gemm_f32_workspace_bytes(b.n_tokens, 2 * di, meta.hidden), ic_gemm_f32_workspace_bytes(b.n_tokens, meta.hidden, di)});
            }
            f32 = std::max(f32, ic_gemm_f32_workspace_bytes(b.n_want, meta.vocab, meta.hidden));
        }
        w.f32_parts = take((size_t)f32);
        if (device_table && b.decode_rows_identity) {      // (what any smaller step needs too: recorded steps share one workspace)
            const int rows = std::min(b.n_tokens, kChainMaxRows);
            w.chain = take(chain_scratch_bytes(chain_shape(), rows, meta.n_entries));
        }
        w.total = o;
        return w;
    }
    // out[M, N] = alpha * a w^T: the few-row product, or what ic_product takes.
    int linear(const void* a, int lda, const void* w, void* out, int out_dtype, int M, int N, int K, float alpha,
               const Deferred* rows, void* f32_parts, void* lib_ws, long long lib_ws_bytes, hipStream_t stream) const {
        if (ic_rule_own_product(meta.dtype, meta.dtype, out_dtype, M)) {
            IcRowFactor rf{};
            if (rows) rf = IcRowFactor{rows->sumsq, rows->parts, rows->width, rows->eps};
            return ic_gemm_nt(a, IC_BF16, w, IC_BF16, out, out_dtype, M, N, K, lda, K, N, alpha, 0, rows ? &rf : nullptr,
                              nullptr, stream);
        }
        if (rows) return IC_ERR_ARG;      // half-normed rows exist only where the few-row product runs
        if (meta.dtype == IC_F32)
            return ic_product_f32(a, w, out, M, N, K, lda, K, N, alpha, f32_parts, ic_gemm_f32_workspace_bytes(M, N, K), lib_ws, lib_ws_bytes, stream);
        return ic_product(a, meta.dtype, w, out, out_dtype, M, N, K, lda, K, N, alpha, lib_ws, lib_ws_bytes, stream);
    }

    // Float32 products of many rows in parts: slices of K where the product runs in parts of all rows at once, else 0 (then `linear` it is).
    int whole_f32(const void* a, const void* w, const void* out, int M, int N, int K, const void* parts) const {
        return meta.dtype == IC_F32 ? ic_gemm_f32_whole(a, w, out, M, N, K, K, K, N, parts, ic_gemm_f32_workspace_bytes(M, N, K)) : 0;
    }
    // Whether ic_norm_parts_f32 takes a norm (ic_add_rmsnorm takes any weight).
    bool norm_in_parts(const IcNorm& norm) const { return ic_norm_parts_f32_supported(meta.hidden) && !((uintptr_t)norm.weight & 15); }
    // Into the residual stream, with slices that the norm after it adds up (slices > 1): those lie behind the K columns' parts, and the norm's parts must not reach them.
    bool leaves_slices(int slices, int K, const IcNorm& norm) const { return slices > 1 && meta.hidden <= K && norm_in_parts(norm); }

    // 17..64 rows (and 13..16 long ones) into the residual stream: x += alpha * (a w^T), out = rmsnorm(x) * weight, through the sliced
    // product and the kernel that sums the slices.
    int tail_in_slices(const void* a, int K, const void* w, float* parts, float* x, float alpha, const float* weight, float eps,
                       void* out, int T, hipStream_t stream) const {
        const int d = meta.hidden;
        const int slices = ic_gemm_splitk_slices(d, K);
        const int st = ic_gemm_splitk(a, w, parts, T, d, K, K, K, slices, stream);
        if (st) return st;
        return ic_splitk_add_rmsnorm(parts, slices, T, x, alpha, weight, out, d, eps, nullptr, 0.f, nullptr, 0.f, stream);
    }

    int forward(const IcStepBatch& b, void* workspace, long long workspace_bytes, void* lib_ws, long long lib_ws_bytes,
                float* logits, hipStream_t stream, int absent = 0, int tries = kChainTries) {
        error.clear();
        const int T = b.n_tokens, d = meta.hidden, dt = meta.dtype, ps = meta.page_size;
        if (T <= 0) return IC_OK;
        if (b.n_requests <= 0 || b.n_want < 0 || b.n_decode_rows < 0 || b.n_prefill_tiles < 0 || !b.tokens || !b.positions ||
            !b.token_req || (b.n_want > 0 && (!logits || !b.want_rows)))
            return fail(IC_ERR_ARG, "the batch description", -1);
        const Workspace ws = layout(b);
        if (!workspace || workspace_bytes < (long long)ws.total) return fail(IC_ERR_ARG, "the workspace (too small)", -1);
        char* base = (char*)workspace;
        float* x = (float*)(base + ws.residual);
        void* normed = base + ws.normed;
        void* qkv = base + ws.qkv;
        void* attn_out = base + ws.attn_out;
        void* f32_parts = base + ws.f32_parts;
        const int parts = ic_gemm_nt_residual_parts(d);
        int st;

        const bool chain = takes_chain(b, workspace);
        if (!chain) {
            st = ic_embed(b.tokens, meta.embed_table, dt, x, T, d, meta.embed_scale, stream);
            if (st) return fail(st, "the embedding gather", -1);
        }

        const int* decode_rows = b.decode_rows_identity ? nullptr : b.decode_rows;
        bool ordered = !b.decode_rows_identity;      // a list of the caller's has the longest rows first

        // what the residual stream still owes when a layer starts
        enum { NONE, BRANCH, DEFERRED, NORMED } owed = NONE;      // NORMED: the add and the whole norm are done, `normed` holds the rows
        const void* branch = nullptr;
        float branch_alpha = 0.f;
        int branch_slices = 1;                       // of the float32 product that left them for the norm to add
        Deferred def;
        // Float32: x += alpha * (the sum of the slices y), normed = its norm, with normed's parts where the product behind it takes them.
        bool in_parts = false;                       // f32_parts holds the parts of the rows that the next product reads
        auto add_norm = [&](const void* y, int slices, float alpha, const IcNorm& norm, int next_slices) {
            in_parts = next_slices > 0 && norm_in_parts(norm);
            if (in_parts || slices > 1)
                return ic_norm_parts_f32(x, (const float*)y, slices, alpha, norm.weight, (float*)normed, in_parts ? f32_parts : nullptr, T, d, norm.eps, stream);
            return ic_add_rmsnorm(x, y, dt, alpha, norm.weight, normed, dt, T, d, norm.eps, stream);
        };
        // a product of these rows, the parts there or not; keep: its slices are left
        auto product = [&](const void* a, const void* w, void* out, int N, int K, int slices, bool keep) {
            const bool ready = in_parts;
            in_parts = false;
            if (slices > 0) return ic_gemm_f32_between(a, w, out, T, N, K, K, K, N, f32_parts, ic_gemm_f32_workspace_bytes(T, N, K), ready, keep, stream);
            return linear(a, K, w, out, dt, T, N, K, 1.0f, nullptr, f32_parts, lib_ws, lib_ws_bytes, stream);
        };

        if (chain) {
            const IcRunEntry& e = entries[0];
            const IcLayer& l = layers[e.layer];
            const IcAttention& A = l.attention;
            if (!b.group_tables[e.group] || !b.group_slots[e.group]) return fail(IC_ERR_ARG, "the cache group of the entry", 0);
            if (b.max_position >= A.max_positions) return fail(IC_ERR_ARG, "a position beyond the rotary tables", 0);
            ChainStep c{device_table, meta.n_entries, T, A.softmax_scale, l.residual_scale, l.mixer_norm.eps, l.ffn_norm.eps, meta.embed_scale,
                        b.tokens, b.positions, b.group_slots[e.group], b.token_req, b.group_tables[e.group], b.group_table_stride[e.group], A.cos, A.sin,
                        meta.embed_table, l.mixer_norm.weight, x, base + ws.chain, base + ws.ffn_tail, (float*)(base + ws.ffn_sumsq), gave_up, tries};
            st = chain_launch(chain_shape(), c, absent, stream);
            if (st) return fail(st, "the layers in one launch", 0);
            def = Deferred{base + ws.ffn_tail, (const float*)(base + ws.ffn_sumsq), chain_sumsq_parts(chain_shape()), d, meta.final_norm.eps};
            owed = DEFERRED;
        }
        const int last = chain ? -1 : meta.n_entries - 1;
        for (int i = 0; i <= last; ++i) {
            const IcRunEntry& e = entries[i];
            const IcLayer& L = layers[e.layer];
            const IcAttention& A = L.attention;
            if (e.group < 0 || e.group >= meta.n_groups || !b.group_tables[e.group]) return fail(IC_ERR_ARG, "the cache group of the entry", i);
            // the norm that whoever runs next applies first, if its rows may reach it half done
            const IcNorm* succ = nullptr;
            const float* succ_weight = nullptr;
            if (i < last) { succ = &layers[entries[i + 1].layer].mixer_norm; succ_weight = succ->weight; }
            else if (b.want_rows_identity) { succ = &meta.final_norm; succ_weight = meta.final_norm_scaled; }

            const int qkv_width = (A.n_heads + 2 * (A.shared_kv ? 0 : A.n_kv_heads)) * A.head_dim;
            const int qkv_slices = whole_f32(normed, A.w_qkv, qkv, T, qkv_width, d, f32_parts);

            // ---- norm before the mixer -------------------------------------------------------------
            const Deferred* h_def = nullptr;
            if (owed == DEFERRED) h_def = &def;
            else if (owed == NORMED) {
            } else if (owed == NONE) {
                st = ic_rmsnorm(x, nullptr, L.mixer_norm.weight, normed, dt, T, d, L.mixer_norm.eps, 1.0f, stream);
                if (st) return fail(st, "the norm before attention", i);
            } else {
                st = add_norm(branch, branch_slices, branch_alpha, L.mixer_norm, qkv_slices);
                if (st) return fail(st, "the residual add and norm before attention", i);
            }
            const void* h = h_def ? h_def->values : normed;

            // ---- attention: QKV, rotary, cache write -------------------------------------------------
            const int nkv = (A.shared_kv || !e.writes_cache) ? 0 : A.n_kv_heads;
            const int width = qkv_width;
            const int* slots = b.group_slots[e.group];
            if (A.rot_dim > 0 && b.max_position >= A.max_positions) return fail(IC_ERR_ARG, "a position beyond the rotary tables", i);
            if (nkv > 0 && !slots) return fail(IC_ERR_ARG, "the cache slots of the entry's group", i);
            const bool fused_qkv = ic_rule_qkv_fused(dt, T, d, d, d, A.head_dim, A.rot_dim, nkv, h_def != nullptr) != 0;
            IcRowFactor rf{};
            if (h_def) rf = IcRowFactor{h_def->sumsq, h_def->parts, h_def->width, h_def->eps};
            if (fused_qkv) {
                st = ic_gemm_qkv_rope(h, A.w_qkv, qkv, T, d, d, d, width, b.positions, slots, A.cos, A.sin, e.k_cache, e.v_cache,
                                      A.n_heads, nkv, A.head_dim, ps, h_def ? &rf : nullptr, stream);
                if (st) return fail(st, "the QKV product with rotary and cache write", i);
            } else if (!h_def && ic_rule_qkv_tiles(dt, h, A.w_qkv, qkv, T, d, d, d, width, A.cos, A.sin, e.k_cache, e.v_cache, A.n_heads, nkv,
                                                   A.head_dim, A.rot_dim, ps)) {
                st = ic_gemm_tiles_rope(h, A.w_qkv, qkv, T, d, d, d, width, b.positions, slots, A.cos, A.sin, e.k_cache, e.v_cache, A.n_heads, nkv,
                                        A.head_dim, ps, stream);
                if (st) return fail(st, "the QKV product with rotary and cache write, in tiles", i);
            } else {
                st = h_def ? linear(h, d, A.w_qkv, qkv, dt, T, width, d, 1.0f, h_def, f32_parts, lib_ws, lib_ws_bytes, stream)
                           : product(h, A.w_qkv, qkv, width, d, qkv_slices, false);
                if (st) return fail(st, "the QKV product", i);
                if (A.rot_dim > 0 || nkv > 0) {
                    st = ic_rope_kv_write(qkv, dt, b.positions, A.rot_dim > 0 ? A.cos : nullptr, A.rot_dim > 0 ? A.sin : nullptr,
                                          nkv > 0 ? e.k_cache : nullptr, nkv > 0 ? e.v_cache : nullptr, nkv > 0 ? slots : nullptr, T,
                                          width, A.n_heads, nkv, A.head_dim, A.rot_dim, ps, stream);
                    if (st) return fail(st, "rotary and cache write", i);
                }
            }

            // ---- attention over the cache ---------------------------------------------------------------
            const int* tables = b.group_tables[e.group];
            const int bts = b.group_table_stride[e.group];
            const int ow = A.n_heads * A.head_dim;
            const int n_dec = b.n_decode_rows, n_tiles = b.n_prefill_tiles;
            const int attn = ic_rule_attention(dt, A.head_dim, ps, n_dec, n_tiles);
            const bool use_dec = (attn & IC_ATTN_SINGLE_TOKENS) != 0, use_pre = (attn & IC_ATTN_PORTIONS) != 0;
            if (attn == IC_ATTN_GENERAL) {
                st = ic_attn_generic(qkv, width, attn_out, ow, dt, e.k_cache, e.v_cache, tables, bts, b.token_req, b.positions, T,
                                     A.n_heads, A.n_kv_heads, A.head_dim, ps, A.softmax_scale, A.window, stream);
                if (st) return fail(st, "attention (general kernel)", i);
            } else if (use_dec && use_pre && decode_rows &&
                       ic_rule_attention_together(dt, A.n_heads, A.n_kv_heads, A.head_dim, ps, bts, n_dec, n_tiles, tiles_end(b), A.window,
                                                  tile_parts_for(b, A, nullptr), meta.compute_units)) {
                int part_len = 0;
                const int parts = mixed_parts_for(b, A, &part_len);
                st = ic_attn_mixed(qkv, width, attn_out, ow, dt, e.k_cache, e.v_cache, tables, bts, decode_rows, b.token_req, b.positions,
                                   (float*)(base + ws.part_acc), (float*)(base + ws.part_ml), n_dec, splits_for(b, A), b.prefill_tiles, n_tiles, A.n_heads,
                                   A.n_kv_heads, A.head_dim, ps, A.softmax_scale, A.window, parts, part_len, (float*)(base + ws.tile_parts),
                                   ic_attn_prefill_scratch_floats(n_tiles, A.n_heads, A.head_dim, parts), meta.attention_counters, stream);
                if (st) return fail(st, "attention of single tokens and prompt portions", i);
            } else {
                if (use_dec) {
                    const int n_split = splits_for(b, A);
                    if (!ordered && ic_attn_decode_wants_order(n_dec, A.n_kv_heads, n_split, meta.compute_units)) {
                        decode_rows = (int*)(base + ws.decode_order);
                        st = ic_attn_decode_order(b.positions, (int*)(base + ws.decode_order), n_dec, stream);
                        if (st) return fail(st, "the order of the single tokens", i);
                        ordered = true;
                    }
                    st = ic_attn_decode(qkv, width, attn_out, ow, dt, e.k_cache, e.v_cache, tables, bts,
                                        decode_rows, b.token_req, b.positions,
                                        (float*)(base + ws.part_acc), (float*)(base + ws.part_ml), n_dec, A.n_heads, A.n_kv_heads,
                                        A.head_dim, ps, A.softmax_scale, A.window, n_split, stream);
                    if (st) return fail(st, "attention of single tokens", i);
                }
                if (use_pre) {
                    int part_len = 0;
                    const int parts = tile_parts_for(b, A, &part_len);
                    st = ic_attn_prefill_split(qkv, width, attn_out, ow, dt, e.k_cache, e.v_cache, tables, bts, b.prefill_tiles,
                                               n_tiles, A.n_heads, A.n_kv_heads, A.head_dim, ps, A.softmax_scale, A.window, 0, parts,
                                               part_len, (float*)(base + ws.tile_parts),
                                               ic_attn_prefill_scratch_floats(n_tiles, A.n_heads, A.head_dim, parts),
                                               meta.attention_counters, stream);
                    if (st) return fail(st, "attention of prompt portions", i);
                }
            }

            // ---- O projection, residual add, norm before the feed-forward --------------------------------
            const int di = L.ffn.intermediate;
            void* act = base + ws.act;
            const int down_slices = whole_f32(act, L.ffn.w_down, base + ws.ffn_out, T, d, di, f32_parts);
            const int gate_up_slices = whole_f32(normed, L.ffn.w_gate_up, base + ws.gate_up, T, 2 * di, d, f32_parts);
            Deferred mid;
            const Deferred* g_def = nullptr;
            const int o_tail = ic_rule_tail(dt, T, d, ow, ow, ow);
            if (o_tail == IC_TAIL_SLICES) {
                st = tail_in_slices(attn_out, ow, A.w_o, (float*)(base + ws.tail_parts), x, L.residual_scale, L.ffn_norm.weight,
                                    L.ffn_norm.eps, normed, T, stream);
                if (st) return fail(st, "the O product in slices with residual add and norm", i);
            } else if (o_tail == IC_TAIL_SPLIT_NORM) {
                IcResidualNorm tail{x, d, L.ffn_norm.weight, L.residual_scale, (float*)(base + ws.mixer_sumsq), parts};
                st = ic_gemm_nt(attn_out, IC_BF16, A.w_o, IC_BF16, base + ws.mixer_tail, IC_BF16, T, d, ow, ow, ow, d, 1.0f, 2, nullptr,
                                &tail, stream);
                if (st) return fail(st, "the O product with residual add", i);
                mid = Deferred{base + ws.mixer_tail, (const float*)(base + ws.mixer_sumsq), parts, d, L.ffn_norm.eps};
                g_def = &mid;
            } else {
                const int o_slices = whole_f32(attn_out, A.w_o, base + ws.mixer_out, T, d, ow, f32_parts);
                const bool keep = leaves_slices(o_slices, ow, L.ffn_norm);
                st = product(attn_out, A.w_o, base + ws.mixer_out, d, ow, o_slices, keep);
                if (st) return fail(st, "the O product", i);
                st = add_norm(keep ? (char*)f32_parts + ic_gemm_f32_parts_bytes(T, ow) : base + ws.mixer_out, keep ? o_slices : 1, L.residual_scale, L.ffn_norm, gate_up_slices);
                if (st) return fail(st, "the residual add and norm before the feed-forward", i);
            }
            const void* g = g_def ? g_def->values : normed;

            // ---- feed-forward ----------------------------------------------------------------------------------
            if (ic_rule_gate_up_fused(dt, T, d, d, d, g_def != nullptr)) {
                IcRowFactor gf{};
                if (g_def) gf = IcRowFactor{g_def->sumsq, g_def->parts, g_def->width, g_def->eps};
                st = ic_gemm_nt(g, IC_BF16, L.ffn.w_gate_up, IC_BF16, act, IC_BF16, T, 2 * di, d, d, d, di, 1.0f, 1, g_def ? &gf : nullptr,
                                nullptr, stream);
                if (st) return fail(st, "the gate/up product with SwiGLU", i);
            } else if (ic_rule_gate_up_tiles(dt, g, L.ffn.w_gate_up, act, T, 2 * di, d, d, d, di)) {
                st = ic_gemm_tiles(g, L.ffn.w_gate_up, act, T, 2 * di, d, d, d, di, 1, stream);
                if (st) return fail(st, "the gate/up product with SwiGLU, in tiles", i);
            } else {
                st = product(g, L.ffn.w_gate_up, base + ws.gate_up, 2 * di, d, gate_up_slices, false);
                if (st) return fail(st, "the gate/up product", i);
                in_parts = down_slices > 0;
                st = in_parts ? ic_swiglu_parts_f32((const float*)(base + ws.gate_up), (float*)act, f32_parts, T, di, stream)
                              : ic_swiglu(base + ws.gate_up, act, dt, T, di, stream);
                if (st) return fail(st, "SwiGLU", i);
            }
            const int down_tail = succ ? ic_rule_tail(dt, T, d, di, di, di) : IC_TAIL_PLAIN;
            if (down_tail == IC_TAIL_SLICES) {
                st = tail_in_slices(act, di, L.ffn.w_down, (float*)(base + ws.tail_parts), x, L.residual_scale, succ_weight, succ->eps,
                                    normed, T, stream);
                if (st) return fail(st, "the down product in slices with residual add and norm", i);
                owed = NORMED;
            } else if (down_tail == IC_TAIL_SPLIT_NORM) {
                IcResidualNorm tail{x, d, succ_weight, L.residual_scale, (float*)(base + ws.ffn_sumsq), parts};
                st = ic_gemm_nt(act, IC_BF16, L.ffn.w_down, IC_BF16, base + ws.ffn_tail, IC_BF16, T, d, di, di, di, d, 1.0f, 2, nullptr,
                                &tail, stream);
                if (st) return fail(st, "the down product with residual add", i);
                def = Deferred{base + ws.ffn_tail, (const float*)(base + ws.ffn_sumsq), parts, d, succ->eps};
                owed = DEFERRED;
            } else {
                const bool keep = i < last && leaves_slices(down_slices, di, layers[entries[i + 1].layer].mixer_norm);      // (the last one's are added up: the final norm takes the wanted rows only)
                st = product(act, L.ffn.w_down, base + ws.ffn_out, d, di, down_slices, keep);
                if (st) return fail(st, "the down product", i);
                branch = keep ? (const char*)f32_parts + ic_gemm_f32_parts_bytes(T, di) : base + ws.ffn_out;
                branch_slices = keep ? down_slices : 1;
                branch_alpha = L.residual_scale;
                owed = BRANCH;
            }
        }

        // ---- final norm and head, on the wanted rows only -----------------------------------------------------
        if (b.n_want == 0) return IC_OK;
        if (owed == NORMED) {        // every row in order, the final norm (with the logit scale in its weight) applied
            st = linear(normed, d, meta.head_weight, logits, IC_F32, T, meta.vocab, d, 1.0f, nullptr, f32_parts, lib_ws, lib_ws_bytes, stream);
            if (st) return fail(st, "the head product", -1);
            return IC_OK;
        }
        if (owed == DEFERRED) {      // every row in order, the final norm half done: its row factors go into the product
            st = linear(def.values, d, meta.head_weight, logits, IC_F32, T, meta.vocab, d, 1.0f, &def, f32_parts, lib_ws, lib_ws_bytes, stream);
            if (st) return fail(st, "the head product", -1);
            return IC_OK;
        }
        if (owed == BRANCH) {
            st = ic_residual_add(x, branch, dt, branch_alpha, (long long)T * d, stream);
            if (st) return fail(st, "the last residual add", -1);
        }
        void* head_in = base + ws.head_in;
        st = ic_rmsnorm(x, b.want_rows, meta.final_norm.weight, head_in, dt, b.n_want, d, meta.final_norm.eps, meta.logit_scale, stream);
        if (st) return fail(st, "the final norm", -1);
        st = linear(head_in, d, meta.head_weight, logits, IC_F32, b.n_want, meta.vocab, d, 1.0f, nullptr, f32_parts, lib_ws, lib_ws_bytes, stream);
        if (st) return fail(st, "the head product", -1);
        return IC_OK;
    }
};

IC_EXPORT long long ic_decoder_table_bytes(int n_entries) { return n_entries < 0 ? -1 : (long long)(n_entries + 1) * (long long)sizeof(ChainEntry); }

IC_EXPORT int ic_decoder_layer_table(const IcDecoder* decoder, void* host) {
    if (!decoder || !host) return IC_ERR_ARG;
    if (decoder->table.empty()) return 0;
    memcpy(host, decoder->table.data(), decoder->table.size() * sizeof(ChainEntry));
    return 1;
}

IC_EXPORT int ic_decoder_use_layer_table(IcDecoder* decoder, const void* table, int* gave_up) {
    if (!decoder || ((uintptr_t)table & 7) || ((uintptr_t)gave_up & 3) || (table && decoder->table.empty())) return IC_ERR_ARG;
    decoder->device_table = (const ChainEntry*)table;
    decoder->gave_up = table ? gave_up : nullptr;
    return IC_OK;
}

IC_EXPORT const char* ic_decoder_create_error() { return g_create_error.c_str(); }

IC_EXPORT IcDecoder* ic_decoder_create(const IcDecoderMeta* meta, const IcLayer* layers, const IcRunEntry* entries) {
    g_create_error.clear();
    auto bad = [&](const char* what) -> IcDecoder* { g_create_error = what; return nullptr; };
    if (!meta || !layers || !entries) return bad("a null description");
    if (meta->dtype != IC_F32 && meta->dtype != IC_BF16) return bad("dtype must be 0 (float32) or 1 (bfloat16)");
    if (meta->hidden <= 0 || meta->vocab <= 0 || meta->page_size <= 0 || meta->n_layers <= 0 || meta->n_entries <= 0)
        return bad("hidden, vocab, page_size, n_layers and n_entries must be positive");
    if (meta->n_groups <= 0 || meta->n_groups > IC_MAX_CACHE_GROUPS) return bad("n_groups must lie in 1..8");
    if (!meta->embed_table || !meta->head_weight || !meta->final_norm.weight || !meta->final_norm_scaled)
        return bad("embedding table, head weight and final norm weights are needed");
    IcDecoder* d = new IcDecoder;
    d->meta = *meta;
    d->layers.assign(layers, layers + meta->n_layers);
    d->entries.assign(entries, entries + meta->n_entries);
    for (const IcLayer& l : d->layers) {
        const IcAttention& a = l.attention;
        const char* why = nullptr;
        if (a.n_heads <= 0 || a.n_kv_heads <= 0 || a.n_heads % a.n_kv_heads) why = "heads must be a positive multiple of kv heads";
        else if (a.head_dim <= 0 || a.head_dim % 16 || a.head_dim > 512) why = "head size must be a multiple of 16 up to 512";
        else if (a.rot_dim < 0 || a.rot_dim % 2 || a.rot_dim > a.head_dim) why = "rot_dim must be even and at most the head size";
        else if (a.rot_dim > 0 && (!a.cos || !a.sin || a.max_positions <= 0)) why = "rotary tables are needed";
        else if (!a.w_qkv || !a.w_o || !l.mixer_norm.weight || !l.ffn_norm.weight) why = "a layer lacks a weight";
        else if (l.ffn.intermediate <= 0 || !l.ffn.w_gate_up || !l.ffn.w_down) why = "the feed-forward lacks a size or a weight";
        if (why) { delete d; return bad(why); }
        d->max_qkv_width = std::max(d->max_qkv_width, (a.n_heads + 2 * (a.shared_kv ? 0 : a.n_kv_heads)) * a.head_dim);
        d->max_attn_width = std::max(d->max_attn_width, a.n_heads * a.head_dim);
        d->max_intermediate = std::max(d->max_intermediate, l.ffn.intermediate);
    }
    for (const IcRunEntry& e : d->entries) {
        if (e.layer < 0 || e.layer >= meta->n_layers || e.group < 0 || e.group >= meta->n_groups || !e.k_cache || !e.v_cache) {
            delete d;
            return bad("a run-order entry names no layer, no group or no cache planes");
        }
    }
    d->make_table();
    return d;
}

IC_EXPORT void ic_decoder_destroy(IcDecoder* decoder) { delete decoder; }

IC_EXPORT const char* ic_decoder_last_error(const IcDecoder* decoder) { return decoder ? decoder->error.c_str() : "no decoder"; }

IC_EXPORT long long ic_decoder_workspace_bytes(const IcDecoder* decoder, const IcStepBatch* batch) {
    if (!decoder || !batch || batch->n_tokens < 0 || batch->n_want < 0 || batch->n_decode_rows < 0) return -1;
    return (long long)decoder->layout(*batch).total;
}

IC_EXPORT int ic_decoder_forward(IcDecoder* decoder, const IcStepBatch* batch, void* workspace, long long workspace_bytes,
                                 void* library_workspace, long long library_workspace_bytes, float* logits, hipStream_t stream) {
    if (!decoder || !batch) return IC_ERR_ARG;
    return decoder->forward(*batch, workspace, workspace_bytes, library_workspace, library_workspace_bytes, logits, stream);
}

// The same with `absent` of the blocks that a step's layers are dealt to not taking part, as if they found no room.
IC_EXPORT int ic_decoder_forward_absent(IcDecoder* decoder, const IcStepBatch* batch, void* workspace, long long workspace_bytes, void* library_workspace,
                                        long long library_workspace_bytes, float* logits, int absent, hipStream_t stream) {
    if (!decoder || !batch || absent < 0 || absent >= decoder->meta.compute_units) return IC_ERR_ARG;
    return decoder->forward(*batch, workspace, workspace_bytes, library_workspace, library_workspace_bytes, logits, stream, absent);
}

// The same where a block gives up a wait after `tries` questions.
IC_EXPORT int ic_decoder_forward_tries(IcDecoder* decoder, const IcStepBatch* batch, void* workspace, long long workspace_bytes, void* library_workspace,
                                       long long library_workspace_bytes, float* logits, int tries, hipStream_t stream) {
    if (!decoder || !batch || tries < 0) return IC_ERR_ARG;
    return decoder->forward(*batch, workspace, workspace_bytes, library_workspace, library_workspace_bytes, logits, stream, 0, tries);
}

// Whether a step runs its layers in one launch.
IC_EXPORT int ic_decoder_takes_chain_at(const IcDecoder* decoder, const IcStepBatch* batch, const void* workspace) { return decoder && batch ? decoder->takes_chain(*batch, workspace) : 0; }
IC_EXPORT int ic_decoder_takes_chain(const IcDecoder* decoder, const IcStepBatch* batch) { return ic_decoder_takes_chain_at(decoder, batch, nullptr); }

// ---- the key split of single-token rows --------------------------------------------------------------------------
// One split writes the result itself; more cost a second kernel.  A rule by a model of the two kernels' time, one for each way of walking the
// keys (one query head per kv head: a wave walks keys with vector instructions; grouped query heads: on the matrix cores); a step's rows
// are taken to be all as long as the longest.  A split never gets fewer than 64 keys.
IC_EXPORT int ic_attn_decode_splits(int n_decode_rows, int n_heads, int n_kv_heads, int head_dim, int elem_bytes, int window,
                                    int max_context, int matrix_cores, int compute_units) {
    const int keys = std::max(1, window > 0 ? std::min(max_context, window) : max_context);
    const long long base = std::max(1LL, (long long)n_decode_rows * n_kv_heads);
    const double cu = compute_units > 0 ? compute_units : 256;
    const int s_max = std::max(1, std::min(64, keys / 64));
    if (matrix_cores) {
        // The grouped-query kernel: the same kind of model as below with constants of its own, fitted to an earlier, slower chain per key tile, and a
        // price of its own for one split of eight waves, whose chain is half as long.  Measured with the present kernel over 1,324 shapes of
        // equal and 1,148 of ragged rows (the shortest a third or a twelfth of the longest; 1..64 rows of 1..8 kv heads with 2..16 query heads each,
        // head sizes 64 and 128, 258..16,400 keys) the count it picks loses 2.3 % to the best one on average, where one split may have eight waves
        // 2.2 (4.4 with four waves' price: it split too early; 12 rows of 24:8 heads over 700 keys: one split 8.2 us, 5 splits 10.4); most, up to 56 %, on
        // rows of very different lengths, where more splits even out what the longest row costs, which the rule does not know.
        if (keys <= 256) return 1;
        const double stream_us = (double)base * keys * std::max(1, head_dim) * 2.0 * std::max(1, elem_bytes) / (6.42e6 * cu / 256.0);
        const double group = (double)std::max(1, n_heads) / std::max(1, n_kv_heads);
        const bool eight = ic_attn_decode_waves(head_dim, (int)std::min(base, 1LL << 30), 1) == 8;
        int best = 1;
        double best_cost = 0.0;
        for (int s = 1; s <= s_max; ++s) {
            const double x = (double)base * s / cu;
            const double lost = 1.0 + (x > 1.0 ? 0.185 : 0.801) * (std::ceil(x) / x - 1.0);
            double cost = 1.882 + 5.201 / s + lost * stream_us;
            if (s > 1) cost += 6.632 + 0.153 * x * group;
            else if (eight) cost = 6.5 + 3.75 * keys / 1024.0 + 0.75 * stream_us;
            if (s == 1 || cost < best_cost) { best_cost = cost; best = s; }
        }
        return best;
    }
    // One head per wave: the split count with the least cost by a model of the two kernels' time in microseconds, fitted
    // to sweeps over 1..32 rows, 8..36 heads of 64 and 128, 600..16,500 keys with caches that do not fit the last-level
    // cache (on 370 shapes it loses 1.5 % against the best count on average, the rule of thumb it replaces 6 %):
    //   the bytes of keys and values at the rate the kernel streams them when every compute unit is busy,
    //   times what is lost when the last round of blocks fills the units only in part (x blocks a unit; less is lost
    //   below one block a unit, where a block's own latency sets the time),
    //   times what is lost when a block's share of the keys is not a whole number of its loop's 256-key rounds,
    //   plus a start-up cost that shrinks with shorter blocks, plus, with more than one split, the second kernel, its
    //   work per split and the partial results per block.
    const double stream_us = (double)base * keys * std::max(1, head_dim) * 2.0 * std::max(1, elem_bytes) / (6.631e6 * cu / 256.0);
    int best = 1;
    double best_cost = 0.0;
    for (int s = 1; s <= s_max; ++s) {
        const double x = (double)base * s / cu;
        double lost = 1.0 + (x > 1.0 ? 0.494 : 0.347) * (std::ceil(x) / x - 1.0);
        const int per = (keys + s - 1) / s;
        lost *= 1.0 + 0.299 * ((double)((per + 255) / 256 * 256) * s / keys - 1.0);
        double cost = 4.757 / s + lost * stream_us;
        if (s > 1) cost += 5.533 + 0.193 * s + 0.38 * x;
        if (s == 1 || cost < best_cost) { best_cost = cost; best = s; }
    }
    return best;
}

// ---- a batch given as host arrays ------------------------------------------------------------------------------------
namespace {

inline long long align4(long long n) { return (n + 3) & ~3LL; }

struct HostLayout {
    long long tokens, positions, token_req, want_rows, decode_rows, tiles, slots[IC_MAX_CACHE_GROUPS], tables[IC_MAX_CACHE_GROUPS], total;
    int n_want, n_decode, n_tiles, stride[IC_MAX_CACHE_GROUPS];
};

bool host_layout(const IcDecoder& dec, const IcHostBatch& b, HostLayout& h) {
    if (b.n_tokens <= 0 || b.n_requests <= 0 || !b.tokens || !b.req_lens || !b.req_pos || !b.tables || !b.table_len || b.tile_rows <= 0)
        return false;
    long long sum = 0;
    h.n_want = h.n_decode = h.n_tiles = 0;
    for (int r = 0; r < b.n_requests; ++r) {
        const int n = b.req_lens[r];
        if (n <= 0 || b.req_pos[r] < 0) return false;
        sum += n;
        if (b.want_count) h.n_want += b.want_count[r];
        if (n == 1) ++h.n_decode;
        else h.n_tiles += (n + b.tile_rows - 1) / b.tile_rows;
    }
    if (sum != b.n_tokens || (h.n_want > 0 && !b.want)) return false;
    const long long T = b.n_tokens;
    long long o = 0;
    auto take = [&](long long n) { const long long at = o; o += align4(n); return at; };
    h.tokens = take(T); h.positions = take(T); h.token_req = take(T);
    h.want_rows = take(h.n_want); h.decode_rows = take(h.n_decode); h.tiles = take(4LL * h.n_tiles);
    const int ps = dec.meta.page_size;
    for (int g = 0; g < dec.meta.n_groups; ++g) {
        int longest = 1;
        for (int r = 0; r < b.n_requests; ++r) {
            const int len = b.table_len[g * b.n_requests + r];
            if (len < (b.req_pos[r] + b.req_lens[r] + ps - 1) / ps || !b.tables[g * b.n_requests + r]) return false;
            longest = std::max(longest, len);
        }
        h.stride[g] = longest;
        h.slots[g] = take(T);
        h.tables[g] = take((long long)b.n_requests * longest);
    }
    h.total = o;
    return true;
}

}  // namespace

IC_EXPORT long long ic_decoder_step_ints(const IcDecoder* decoder, const IcHostBatch* batch) {
    HostLayout h;
    if (!decoder || !batch || !host_layout(*decoder, *batch, h)) return -1;
    return h.total;
}

IC_EXPORT int ic_decoder_pack(const IcDecoder* decoder, const IcHostBatch* batch, int* staging, const int* device_ints,
                              long long n_ints, IcStepBatch* out) {
    HostLayout h;
    if (!decoder || !batch || !staging || !device_ints || !out || !host_layout(*decoder, *batch, h) || n_ints < h.total) return IC_ERR_ARG;
    const IcHostBatch& b = *batch;
    const int ps = decoder->meta.page_size, R = b.n_requests;
    struct Row { int pos, row; };
    struct Tile { int req, row, rows, pos; };
    std::vector<Row> dec;
    std::vector<Tile> tiles;
    dec.reserve(h.n_decode);
    tiles.reserve(h.n_tiles);
    int row0 = 0, w = 0, max_pos = 0, max_tile = 0, max_ctx = 0;
    const int* want = b.want;
    bool identity = h.n_want == b.n_tokens;
    for (int r = 0; r < R; ++r) {
        const int n = b.req_lens[r], p0 = b.req_pos[r];
        for (int i = 0; i < n; ++i) {
            staging[h.tokens + row0 + i] = b.tokens[row0 + i];
            staging[h.positions + row0 + i] = p0 + i;
            staging[h.token_req + row0 + i] = r;
        }
        const int nw = b.want_count ? b.want_count[r] : 0;
        for (int i = 0; i < nw; ++i) {
            if (want[i] < 0 || want[i] >= n) return IC_ERR_ARG;
            identity = identity && (row0 + want[i] == w);
            staging[h.want_rows + w++] = row0 + want[i];
        }
        want += nw;
        if (n == 1) { dec.push_back(Row{p0, row0}); max_ctx = std::max(max_ctx, p0 + 1); }
        else {
            for (int o = 0; o < n; o += b.tile_rows) tiles.push_back(Tile{r, row0 + o, std::min(b.tile_rows, n - o), p0 + o});
            max_tile = std::max(max_tile, p0 + n - 1);
        }
        max_pos = std::max(max_pos, p0 + n - 1);
        for (int g = 0; g < decoder->meta.n_groups; ++g) {
            const int* table = b.tables[g * R + r];
            const int len = b.table_len[g * R + r], stride = h.stride[g];
            for (int i = 0; i < n; ++i) staging[h.slots[g] + row0 + i] = table[(p0 + i) / ps] * ps + (p0 + i) % ps;
            int* dst = staging + h.tables[g] + (long long)r * stride;
            for (int j = 0; j < len; ++j) dst[j] = table[j] > 0 ? table[j] : 0;     // pages given back are never read; keep the index valid
            for (int j = len; j < stride; ++j) dst[j] = 0;
        }
        row0 += n;
    }
    // tiles that see the most keys go first, so the longest blocks do not form the tail; likewise the single tokens,
    // unless all rows are single tokens and the kernel takes the rows as they lie
    std::stable_sort(tiles.begin(), tiles.end(), [](const Tile& a, const Tile& c) { return a.pos + a.rows > c.pos + c.rows; });
    if ((int)dec.size() < b.n_tokens) std::stable_sort(dec.begin(), dec.end(), [](const Row& a, const Row& c) { return a.pos > c.pos; });
    for (size_t i = 0; i < dec.size(); ++i) staging[h.decode_rows + i] = dec[i].row;
    for (size_t i = 0; i < tiles.size(); ++i) {
        int* t = staging + h.tiles + 4 * i;
        t[0] = tiles[i].req; t[1] = tiles[i].row; t[2] = tiles[i].rows; t[3] = tiles[i].pos;
    }
    IcStepBatch s{};
    s.n_tokens = b.n_tokens; s.n_requests = R; s.n_want = h.n_want; s.n_decode_rows = (int)dec.size(); s.n_prefill_tiles = (int)tiles.size();
    s.want_rows_identity = identity ? 1 : 0;
    s.decode_rows_identity = (int)dec.size() == b.n_tokens ? 1 : 0;
    s.max_position = max_pos;
    s.max_tile_position = max_tile;
    s.max_context = max_ctx ? ic_rule_context_bucket(max_ctx) : 0;
    s.fixed_decode_splits = b.fixed_decode_splits;
    s.tokens = device_ints + h.tokens; s.positions = device_ints + h.positions; s.token_req = device_ints + h.token_req;
    s.want_rows = device_ints + h.want_rows; s.decode_rows = device_ints + h.decode_rows; s.prefill_tiles = device_ints + h.tiles;
    for (int g = 0; g < decoder->meta.n_groups; ++g) {
        s.group_slots[g] = device_ints + h.slots[g];
        s.group_tables[g] = device_ints + h.tables[g];
        s.group_table_stride[g] = h.stride[g];
    }
    *out = s;
    return IC_OK;
}

IC_EXPORT int ic_decoder_step(IcDecoder* decoder, const IcHostBatch* batch, int* staging, int* device_ints, long long n_ints,
                              void* workspace, long long workspace_bytes, void* library_workspace, long long library_workspace_bytes,
                              float* logits, IcStepBatch* laid_out, hipStream_t stream) {
    IcStepBatch s;
    int st = ic_decoder_pack(decoder, batch, staging, device_ints, n_ints, &s);
    if (st) return decoder ? decoder->fail(st, "laying out the batch", -1) : st;
    const long long need = ic_decoder_step_ints(decoder, batch);
    hipError_t e = hipMemcpyAsync(device_ints, staging, (size_t)need * sizeof(int), hipMemcpyHostToDevice, stream);
    if (e != hipSuccess) return decoder->fail((int)e, "the copy of the step's integers", -1);
    if (laid_out) *laid_out = s;
    return decoder->forward(s, workspace, workspace_bytes, library_workspace, library_workspace_bytes, logits, stream);
}
