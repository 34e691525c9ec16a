// Entry points for tests and sweeps: the few-row products with a variant of their kernels named by the caller, and what kernels choose or compute
// by themselves.  Not part of the interface a caller of the library needs: ic_gemm_nt and ic_gemm_qkv_rope choose for themselves.
// A variant holds for the one call that names it and changes nothing for any other call, thread or engine.
#pragma once
#include "infinicore_infer_engine.h"

#ifdef __cplusplus
extern "C" {
#endif

// ic_gemm_nt with whole_lines == 0: the weights are loaded in operand layout also where whole cache lines through LDS would apply
// (K a multiple of 64, aligned operands); products of 17..32 rows with an epilogue, which exist with whole lines only, are refused.
int ic_gemm_nt_variant(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int c_mode, const IcRowFactor* row_factor, const IcResidualNorm* tail, int whole_lines, hipStream_t stream);
// ic_gemm_qkv_rope with the used weight rows per tile given: 16, 8 or 4 (0: chosen from the number of heads, as ic_gemm_qkv_rope does).
int ic_gemm_qkv_rope_variant(const void* A, const void* W, void* C, int M, int K, int lda, int ldw, int ldc, const int* positions, const int* slots, const float* cos_t, const float* sin_t, void* kcache, void* vcache, int nh, int nkvh, int dh, int page_size, const IcRowFactor* row_factor, int tile_rows, hipStream_t stream);
// The few-row product with the tiling chosen by the caller; nt == 0 selects the SwiGLU variant.
int ic_gemm_nt_cfg(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int nt, int wpb, int unroll, hipStream_t stream);

// Which kernel a product of up to 8 rows with an epilogue takes on a device of `units` compute units.  epi: 1 SwiGLU, 2 rotary and cache write, 3 residual
// add over `blocks` column blocks.  1 and plan[6] = (groups of 8 weight rows a block, lines of 64 k a register stage, waves, token rows through LDS,
// blocks, columns a block) for the kernel of gemm_rows.hip; 0 for the kernels of gemm.hip.
int ic_gemm_rows_plan(int epi, int M, int N, int K, int blocks, int units, int* plan);

// ic_gemm_tiles and ic_gemm_tiles_rope with their tile named by the caller (0..14, the order in gemm_tiles.hip), and the tile that the former chooses by itself (-1: an argument fault).
int ic_gemm_tiles_cfg(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, int mode, int tile, hipStream_t stream);
int ic_gemm_tiles_rope_cfg(const void* A, const void* W, void* C, int M, int K, int lda, int ldw, int ldc, const int* positions, const int* slots, const float* cos_t, const float* sin_t, void* kcache, void* vcache, int nh, int nkvh, int dh, int page_size, int tile, hipStream_t stream);
int ic_gemm_tiles_plan(int M, int N, int K, int mode);
// The same, and ic_gemm_tiles_pays, for a device or partition of `units` compute units.
int ic_gemm_tiles_plan_on(int M, int N, int K, int mode, int units);
int ic_gemm_tiles_pays_on(int M, int N, int K, int mode, int units);
// Notes what timing a product found (ic_product_tune does).
void ic_product_timing(int M, int N, int K, int lda, int ldw, int ldc, int tiles);
void ic_product_f32_timing(int M, int N, int K, int lda, int ldw, int ldc, int own);

// ic_gemm_f32 with its shape (0..14, the order in gemm_f32.hip) and number of slices of K (1..4) named by the caller; the shape that it chooses by itself on a device of
// `units` compute units (-1: an argument fault) and the slices, and ic_gemm_f32_pays for such a device.
int ic_gemm_f32_cfg(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int shape, int slices, void* workspace, long long workspace_bytes, hipStream_t stream);
int ic_gemm_f32_plan_on(int M, int N, int K, int units, int* slices);
int ic_gemm_f32_pays_on(int M, int N, int K, int units);
// The same with a workspace of that size (ic_gemm_f32_pays: of ic_gemm_f32_workspace_bytes).
int ic_gemm_f32_pays_with(int M, int N, int K, long long workspace_bytes, int units);
// Whether ic_gemm_f32 takes a product of 16-byte aligned operands with this workspace.
int ic_gemm_f32_takes(int M, int N, int K, int lda, int ldw, int ldc, const void* workspace, long long workspace_bytes);

// key / page_size as the kernels of single tokens compute it; -1: an argument fault.
int ic_attn_decode_page_of(int key, int page_size);

// The pieces of a decode step's attention as the kernel of whole layers deals them (decode_chain.hip), six ints each: block, row, kv head, first key, key after the
// last, place; and for every (row, kv head) the blocks from .. to whose pieces are brought together (from > to: a block walks the whole head).  Returns their number.
int ic_decode_chain_pieces(const int* positions, int rows, int kv_heads, int compute_units, int* pieces, int capacity, int* from_to);

// ic_decoder_forward with `absent` of the blocks that a decode step's layers are dealt to not taking part, as if they found no room on the device; with waits for other
// blocks that are given up after `tries` questions; and whether a step runs its layers in one launch (on which the two have no effect where it does not), with that
// workspace or an aligned one.
int ic_decoder_forward_absent(IcDecoder* decoder, const IcStepBatch* batch, void* workspace, long long workspace_bytes, void* library_workspace, long long library_workspace_bytes, float* logits, int absent, hipStream_t stream);
int ic_decoder_forward_tries(IcDecoder* decoder, const IcStepBatch* batch, void* workspace, long long workspace_bytes, void* library_workspace, long long library_workspace_bytes, float* logits, int tries, hipStream_t stream);
int ic_decoder_takes_chain(const IcDecoder* decoder, const IcStepBatch* batch);
int ic_decoder_takes_chain_at(const IcDecoder* decoder, const IcStepBatch* batch, const void* workspace);

// Whether ic_causal_conv runs a thread over a run of tokens (four taps, aligned rows), and whether ic_hc_step's threads send several rounds of a row's
// loads ahead.
int ic_causal_conv_runs(int n_tok, int C, int n_requests);
int ic_hc_step_loads_ahead(int S, int T, int d, int read);

#ifdef __cplusplus
}
#endif
