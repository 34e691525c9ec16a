// Attention of a mixed step in one launch: blocks of single tokens (attn_decode_blocks.h) and of prompt tiles (attn_prefill_mfma.h) side by side.
//
// One after the other each kernel has a tail in which most of the chip runs dry (its longest walk over the keys), and the two are bound by
// different things: single tokens by the chain of one tile of keys in a wave and by memory, prompt tiles by softmax and matrix products.  Here the
// single tokens' blocks come first, longest row first, and the prompt tiles' blocks fill the units beside and after them.
#include "attn_decode_blocks.h"
#include "attn_prefill_mfma.h"
#include "infinicore_infer_variants.h"

namespace {

struct MixedArgs {
    const uint16_t* q;
    int q_stride;
    uint16_t* out;
    int out_stride;
    const uint16_t* kcache;
    const uint16_t* vcache;
    const int* block_tables;
    int bt_stride, nh, nkvh, page_size, page_shift, window;
    float scale, scale_log2e;
    // single tokens
    const int* tok_list;
    const int* token_req;
    const int* positions;
    float* part_acc;
    float* part_ml;
    int n_tok, nsplit;
    // prompt tiles
    const int4* tiles;
    int n_tiles, parts, part_len;
    float* scratch;
    int* counters;
};

// GROUPED: query heads share kv heads
template <int DH, bool GROUPED>
__global__ void __launch_bounds__(256, DH <= 64 ? 3 : 2) attn_mixed_kernel(MixedArgs a, PageDivider div) {
    constexpr int STAGE = prefill_stage_elements<DH, 1>(), TILES = GROUPED ? gqa_tile_elements<DH, 4>() : 0;
    __shared__ __attribute__((aligned(16))) uint16_t stage0[STAGE > TILES ? STAGE : TILES];
    __shared__ __attribute__((aligned(16))) uint16_t stage1[STAGE];
    __shared__ int pages[kPfMaxPages];
    static_assert(kPfMaxPages >= kDecMaxPages && sizeof(uint16_t) * STAGE >= sizeof(float) * 4 * 16 * 2, "room for either block");
    const unsigned singles = (unsigned)(a.n_tok * a.nkvh * a.nsplit);
    if (blockIdx.x < singles) {
        const int split = blockIdx.x % a.nsplit, rest = blockIdx.x / a.nsplit, kvh = rest % a.nkvh, n = rest / a.nkvh;
        uint16_t* const direct = a.nsplit == 1 ? a.out : nullptr;   // one split writes the result itself
        if constexpr (GROUPED)
            gqa_block<DH, true, 4>(a.q, a.q_stride, a.kcache, a.vcache, a.block_tables, a.bt_stride, a.tok_list, a.token_req, a.positions, a.part_acc,
                                   a.part_ml, a.nh, a.nkvh, a.page_size, a.scale, a.window, a.nsplit, div, direct, a.out_stride, split, kvh, n, stage0,
                                   reinterpret_cast<float (*)[16][2]>(stage1), pages);
        else
            split_block<bf16, DH, 1, true>((const bf16*)a.q, a.q_stride, (const bf16*)a.kcache, (const bf16*)a.vcache, a.block_tables, a.bt_stride,
                                           a.tok_list, a.token_req, a.positions, a.part_acc, a.part_ml, a.nh, a.nkvh, a.page_size, a.scale, a.window,
                                           a.nsplit, div, (bf16*)direct, a.out_stride, split, kvh, n, reinterpret_cast<float (*)[1][DH]>(stage0),
                                           reinterpret_cast<float (*)[1][2]>(stage1), pages);
    } else {
        prefill_block<DH, true, 1, true>(a.q, a.q_stride, a.out, a.out_stride, a.kcache, a.vcache, a.block_tables, a.bt_stride, a.tiles, a.n_tiles,
                                         a.nh, a.nkvh, a.page_shift, a.scale_log2e, a.window, a.parts, a.part_len, a.scratch, a.counters,
                                         blockIdx.x - singles, stage0, stage1, pages);
    }
}

}  // namespace

// bfloat16, pages of 64 tokens and more (a power of two), block tables that fit the kernels' LDS.
IC_EXPORT int ic_attn_mixed_supported(int dtype, int nh, int nkvh, int dh, int page_size, int bt_stride) {
    return dtype == IC_BF16 && (dh == 64 || dh == 128) && nh > 0 && nkvh > 0 && nh % nkvh == 0 && page_size >= kPfKeys &&
           (page_size & (page_size - 1)) == 0 && bt_stride > 0 && bt_stride <= kDecMaxPages && bt_stride <= kPfMaxPages;
}

// Into how many parts the tiles' walks are cut here, and key tiles per part: as ic_attn_prefill_parts_of_step says for tiles alone, and in two where it
// leaves walks of 12 key tiles and more whole with up to 1.25 blocks a unit, since there two wave groups share such a walk and here there is one.
// Whole against two parts, 40 rows of 100..2,048 keys beside portions of 512 and 463 after 512: 24:8 heads of 64 25.9 -> 25.2 us, 36:36 62.9 -> 60.0,
// 32:2 of 128 41.3 -> 39.4; 6 rows beside a prompt of 1,200: 23.2 -> 20.4, 28.8 -> 24.7, 37.7 -> 36.8.  With 1.5 blocks a unit (32:32 of 128,
// portions of 700 after 600 and 100) 42.1 -> 44.4.
IC_EXPORT int ic_attn_mixed_parts_of_step(int dtype, int n_tiles, int nh, int dh, int max_tile_position, int window, int compute_units, int* part_len) {
    int len = 0, parts = ic_attn_prefill_parts_of_step(dtype, n_tiles, nh, dh, max_tile_position, window, compute_units, &len);
    const long long blocks = (long long)n_tiles * nh;
    if (dtype == IC_BF16 && parts == 1 && len >= 12 && blocks > 0 && blocks <= kPfCounters && (dh == 64 || dh == 128) && 4 * blocks <= 5LL * compute_units) {
        parts = 2;
        len = len > 22 ? (len + 1) / 2 : 11;                // (a shorter walk of the same step stays whole)
    }
    if (part_len) *part_len = len;
    return parts;
}

IC_EXPORT int ic_attn_mixed(const void* q, int q_stride, void* out, int out_stride, int dtype, const void* kcache, const void* vcache,
                            const int* block_tables, int bt_stride, const int* tok_list, const int* token_req, const int* positions, float* part_acc,
                            float* part_ml, int n_tok, int nsplit, const int* tiles, int n_tiles, int nh, int nkvh, int dh, int page_size, float scale,
                            int window, int parts, int part_len, float* scratch, long long scratch_floats, int* counters, hipStream_t stream) {
    if (n_tok <= 0 || n_tiles <= 0 || nsplit <= 0 || nsplit > 64) return IC_ERR_ARG;
    if (!ic_attn_mixed_supported(dtype, nh, nkvh, dh, page_size, bt_stride)) return IC_ERR_UNSUPPORTED;
    if (!q || !out || !kcache || !vcache || !block_tables || !tok_list || !token_req || !positions || !tiles || nkvh > 65535 || nh > 65535 || n_tok > 65535)
        return IC_ERR_ARG;
    if (q_stride % 8 || out_stride % 4 || ((uintptr_t)q & 15) || ((uintptr_t)out & 7) || ((uintptr_t)kcache & 15) || ((uintptr_t)vcache & 15) ||
        ((uintptr_t)tiles & 15)) return IC_ERR_ARG;
    if (nsplit > 1 && (!part_acc || !part_ml)) return IC_ERR_ARG;
    if (parts < 1) parts = 1;
    if (parts > 1 && (part_len < 1 || parts > 64 || (long long)nh * n_tiles > kPfCounters || !scratch || !counters || ((uintptr_t)scratch & 15) ||
                      scratch_floats < ic_attn_prefill_scratch_floats(n_tiles, nh, dh, parts))) return IC_ERR_ARG;
    const long long blocks = (long long)n_tok * nkvh * nsplit + (long long)nh * n_tiles * parts;
    if (blocks > 0x7fffffffLL) return IC_ERR_ARG;
    int page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
    const MixedArgs a{(const uint16_t*)q, q_stride, (uint16_t*)out, out_stride, (const uint16_t*)kcache, (const uint16_t*)vcache, block_tables, bt_stride,
                      nh, nkvh, page_size, page_shift, window, scale, scale * 1.4426950408889634f, tok_list, token_req, positions, part_acc, part_ml,
                      n_tok, nsplit, (const int4*)tiles, n_tiles, parts, part_len, scratch, counters};
    const PageDivider div(page_size);
#define IC_MIXED_LAUNCH(DD, GG) hipLaunchKernelGGL((attn_mixed_kernel<DD, GG>), dim3((unsigned)blocks), dim3(256), 0, stream, a, div)
    const bool grouped = ic_attn_decode_on_matrix_cores(dtype, nh, nkvh) != 0;
    if (dh == 64) { if (grouped) IC_MIXED_LAUNCH(64, true); else IC_MIXED_LAUNCH(64, false); }
    else { if (grouped) IC_MIXED_LAUNCH(128, true); else IC_MIXED_LAUNCH(128, false); }
#undef IC_MIXED_LAUNCH
    const int st = ic_launch_status();
    if (st || nsplit == 1) return st;
    return ic_attn_decode_merge(part_acc, part_ml, tok_list, out, out_stride, dtype, n_tok, nh, dh, nsplit, stream);
}
