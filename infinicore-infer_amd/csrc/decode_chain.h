// All layers of a decode step in one launch (decode_chain.hip), for decoder.hip.
#pragma once
#include "common.h"

constexpr int kChainMaxRows = 8;
constexpr int kChainTries = 1 << 22;

// One run-order entry where it lies on the device; the table has one more than there are entries, whose norm_in is the final norm's weight.
struct ChainEntry {
    const void* w_qkv;
    const void* w_o;
    const void* w_gate_up;
    const void* w_down;
    const float* norm_in;      // of the norm before attention
    const float* norm_mid;     // before the feed-forward
    void* k_cache;
    void* v_cache;
};

// What all entries have in common.
struct ChainShape {
    int hidden, n_heads, n_kv_heads, head_dim, intermediate, page_size, compute_units;
};

struct ChainStep {
    const ChainEntry* entries;
    int n_entries, rows;
    float softmax_scale, residual_scale, eps_in, eps_mid, embed_scale;
    const int *tokens, *positions, *slots, *token_req, *tables;
    int table_stride;
    const float *cos_t, *sin_t;
    const void* embed_table;
    const float* first_norm;   // weight of the first entry's norm before attention
    float* x;                  // float32 residual stream [rows, hidden], left as after the last layer
    void* scratch;             // chain_scratch_bytes
    void* y_out;               // bfloat16 [rows, hidden]: x times the final norm's weight
    float* sumsq_out;          // [parts, 16] sums of squares of x per column block
    int* gave_up;              // set to 1 (null: not) where a wait of a block was given up after `tries` questions
    int tries;
};

// 1: the kernel takes these sizes.  max_keys: an upper bound of the keys that a row sees.
int chain_supported(const ChainShape& s, int rows, int n_entries, int max_keys);
int chain_sumsq_parts(const ChainShape& s);
size_t chain_scratch_bytes(const ChainShape& s, int rows, int n_entries);
// absent: blocks that do not take part (tests).
int chain_launch(const ChainShape& s, const ChainStep& step, int absent, hipStream_t stream);
