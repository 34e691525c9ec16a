// The few-row product's epilogues, and the product of up to 8 rows whose weights go from memory straight into the operand
// registers of the matrix cores (gemm_rows.hip); gemm.hip holds the other kernels of the few-row product and chooses.
#pragma once
#include "common.h"

// What the fused projection + rotary + cache-write epilogue needs beside the product.
struct RopeEpilogue {
    const int* positions;      // [M]
    const int* slots;          // [M] token slot in the cache (page * page_size + offset), < 0: no write
    const float* cos_t;        // [max_pos, dh/2]
    const float* sin_t;
    void* kcache;              // [pages, nkvh, page_size, dh]
    void* vcache;
    int nh, nkvh, dh, page_size;
    int rr;                    // weight rows per tile that are used: 16, 8 or 4 (few heads: smaller tiles make more blocks)
};

// A norm split over two products (M <= 16).  The product BEFORE the norm (EPI == 3) owns the
// residual add: h = x + rscale * (its result), written back to x; it stores y = h * g (g: the
// norm's weight) instead of its result, and per column block the sums of h^2 of every row.  The
// product AFTER the norm takes y as its operand and multiplies row m of its result by
// rsqrt(sum over the column blocks / width + eps): the norm's row factor commutes with the product.
constexpr int kMaxSumParts = 256;
struct NormFuse {
    const float* ss_in;        // [n_parts_in, 16] sums of squares per column block and row; nullptr: rows are normed already
    int n_parts_in;            // <= kMaxSumParts
    float inv_width, eps;
    float* x;                  // EPI == 3: float32 residual stream [M, N], row stride ldx, updated in place
    int ldx;
    const float* g;            // [N]
    float rscale;
    float* ss_out;             // [gridDim.x, 16]
    int act;                   // plain store only: 0 none, else the product (rounded to its type first, as when stored) goes
                               // through an activation: 1 relu(z)^2, 2 gelu_tanh(z), 3 silu(z)
    float glu_limit, glu_slope; // the gated epilogue: limit > 0: the unit with bounded branches instead of up * silu(gate)
};

__device__ __forceinline__ float gemm_act(float z, int act) {
    if (act == 1) { const float r = fmaxf(z, 0.f); return r * r; }
    if (act == 2) return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    return z / (1.0f + expf(-z));
}

// Launches the kernel of gemm_rows.hip when it takes these sizes and is the faster one for them; false: nothing was launched.
// epi: 1 gate/up with the gated unit, 2 rotary and cache write, 3 residual add over `blocks` column blocks.
bool gemm_rows_launch(int epi, const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha,
                      const RopeEpilogue& rope, const NormFuse& nf, int blocks, hipStream_t stream);
