// Attention of prompt portions over the paged cache on the matrix cores: the kernel (its block: attn_prefill_mfma.h), the rules of its launch.
#include "attn_prefill_mfma.h"

template <int DH, bool STAGED, int GROUPS, bool PAGE64>
__global__ void __launch_bounds__(256 * GROUPS, (GROUPS == 1 && DH <= 64) ? 3 : 2)
attn_prefill_mfma_kernel(const uint16_t* __restrict__ q, int q_stride, uint16_t* __restrict__ out, int out_stride,
                         const uint16_t* __restrict__ kcache, const uint16_t* __restrict__ vcache,
                         const int* __restrict__ block_tables, int bt_stride, const int4* __restrict__ tiles,
                         int n_tiles, int nh, int nkvh, int page_shift, float scale_log2e, int window,
                         int parts, int part_len, float* __restrict__ scratch, int* __restrict__ counters) {
    __shared__ __attribute__((aligned(16))) uint16_t stage0[prefill_stage_elements<DH, GROUPS>()];
    __shared__ __attribute__((aligned(16))) uint16_t stage1[prefill_stage_elements<DH, GROUPS>()];
    __shared__ int pages[kPfMaxPages];
    prefill_block<DH, STAGED, GROUPS, PAGE64>(q, q_stride, out, out_stride, kcache, vcache, block_tables, bt_stride, tiles, n_tiles, nh, nkvh,
                                              page_shift, scale_log2e, window, parts, part_len, scratch, counters, blockIdx.x, stage0, stage1, pages);
}

// bfloat16: the kernel above.  float32: the kernel of attn_prefill_f32.hip, in three bfloat16 parts a number (same tiles, one to four key groups a block, walks never cut).
IC_EXPORT int ic_attn_prefill_supported(int dtype, int dh, int page_size) {
    return (dtype == IC_BF16 || dtype == IC_F32) && (dh == 64 || dh == 128) && page_size > 0 && (page_size & (page_size - 1)) == 0;
}

int ic_attn_prefill_f32_launch(const void* q, int q_stride, void* out, int out_stride, const void* kcache, const void* vcache,
                               const int* block_tables, int bt_stride, const int* tiles, int n_tiles, int nh, int nkvh, int dh,
                               int page_shift, float scale, int window, hipStream_t stream);

IC_EXPORT int ic_attn_prefill_tile_rows() { return kPfRows; }
IC_EXPORT int ic_attn_prefill_counter_ints() { return kPfCounters; }

// Floats of scratch memory that a walk cut into `parts` needs: every (tile, head, part) keeps a maximum, a sum and O^T per row.
IC_EXPORT long long ic_attn_prefill_scratch_floats(int n_tiles, int nh, int dh, int parts) {
    if (n_tiles <= 0 || nh <= 0 || parts <= 1 || (dh != 64 && dh != 128)) return 0;
    return (long long)n_tiles * nh * parts * kPfWaveThreads * (2 + dh / 2);
}

// How to cut the walks of a step whose longest query tile sees `max_keys` keys: parts per tile (1: no cut) and key tiles
// per part.  From sweeps over 16..48 heads of 64 and 32..40 of 128, prompts of 300..4,096 tokens and portions of 256..1,024
// after 256..3,584 tokens, against one and two wave groups:
//  * with many blocks, parts pay when walks are long (24 key tiles and more): as many parts as keep about 4.5 blocks a compute
//    unit at head size 64 and 2 at head size 128 (what stays resident there), at most 4, each of 6 key tiles or more; two
//    parts do no better than two wave groups where those run (up to 2 blocks a unit), so they keep that case;
//  * with few blocks (a portion or two beside decoded tokens) shorter walks are cut too: head size 64, up to half a block a
//    unit, from 12 key tiles on into 3 parts (4 from 20 key tiles on when four parts of every block still fit the units at once), and up to 1.25 blocks a unit
//    from 20 key tiles on into 3; head size 128, up to half a block a unit, walks of 8..23 key tiles into 2 parts, and up to a
//    quarter block a unit from 16 key tiles on into 4.  Against two wave groups, portions of 512 tokens after 512..768:
//    24:8 x 64 (96 blocks) 17.6 -> 14.7 and 20.0 -> 17.0 us, 32:2 x 128 (128 blocks) 25.9 -> 22.0 and 29.8 -> 25.1; 256
//    tokens after 1,024: 19.8 -> 13.9 and 29.2 -> 19.9;
//  * portions after a long past gain most (16 heads, 512 tokens after 3,584: 54 -> 26 us; 36 heads: 54 -> 41; 32:2 x 128: 83 -> 52),
//    whole prompts little (36 heads, 2,048 tokens: 43 -> 41 us) or nothing.
IC_EXPORT int ic_attn_prefill_parts(int n_tiles, int nh, int dh, int max_keys, int compute_units, int* part_len) {
    const int longest = (max_keys + kPfKeys - 1) / kPfKeys;
    const long long blocks = (long long)n_tiles * nh, cu = compute_units;
    int len = longest > 0 ? longest : 1, parts = 1;
    if (compute_units > 0 && blocks > 0 && blocks <= kPfCounters && (dh == 64 || dh == 128)) {
        long long p = 1;
        int least = 6;                                      // key tiles a part has at least
        bool few = false;
        if (dh == 64) {
            if (2 * blocks <= cu && longest >= 12) { p = (4 * blocks <= cu && longest >= 20) ? 4 : 3; few = true; }
            else if (4 * blocks <= 5 * cu && longest >= 20) { p = 3; few = true; }
        } else {
            if (4 * blocks <= cu && longest >= 16) { p = 4; few = true; }
            else if (2 * blocks <= cu && longest >= 8 && longest < 24) { p = 2; few = true; }
        }
        if (few) least = 4;
        else if (longest >= 24) {
            const long long room = dh == 64 ? 9LL * cu / 2 : 2LL * cu;
            p = room / blocks;
            p = p > 4 ? 4 : p;
            if (p == 2 && blocks <= 2LL * cu) p = 1;
        }
        p = p > longest / least ? longest / least : p;
        if (p >= 2) {
            parts = (int)p;
            len = (longest + parts - 1) / parts;
            len = len < least ? least : len;
        }
    }
    if (part_len) *part_len = len;
    return parts;
}

// The same question for a step: the largest position of its prompt portions and the mixer's window (0: none) give the most keys a tile sees.
// (float32 walks are never cut.)
IC_EXPORT int ic_attn_prefill_parts_of_step(int dtype, int n_tiles, int nh, int dh, int max_tile_position, int window, int compute_units, int* part_len) {
    int keys = max_tile_position + 1;
    if (dtype != IC_BF16) {
        if (part_len) *part_len = (keys + kPfKeys - 1) / kPfKeys;
        return 1;
    }
    if (window > 0 && window + kPfRows < keys) keys = window + kPfRows;
    return ic_attn_prefill_parts(n_tiles, nh, dh, keys, compute_units, part_len);
}

// tiles: int32 [n_tiles, 4] = (request row of block_tables, first token row, rows <= 128, position of the first row).
// groups: 1 or 2 wave groups per query tile, 0 = chosen from the number of blocks.  parts > 1 (one group only): the grid
// holds `parts` blocks per (tile, head) and a tile's walk is cut into up to that many parts of at least part_len key
// tiles; scratch then holds ic_attn_prefill_scratch_floats(...) floats.
IC_EXPORT int ic_attn_prefill_split(const void* q, int q_stride, void* out, int out_stride, int dtype,
                                    const void* kcache, const void* vcache, const int* block_tables,
                                    int bt_stride, const int* tiles, int n_tiles, int nh, int nkvh, int dh,
                                    int page_size, float scale, int window, int groups, int parts, int part_len,
                                    float* scratch, long long scratch_floats, int* counters, hipStream_t stream) {
    if (n_tiles <= 0) return IC_OK;
    if (!ic_attn_prefill_supported(dtype, dh, page_size)) return IC_ERR_UNSUPPORTED;
    int page_shift = 0;
    while ((1 << page_shift) < page_size) ++page_shift;
    if (nh <= 0 || nkvh <= 0 || nh % nkvh || page_size <= 0 || nh > 65535 || groups < 0 || groups > 2) return IC_ERR_ARG;
    if (dtype == IC_F32)                                  // (groups, parts and scratch do not apply: its walks are never cut)
        return ic_attn_prefill_f32_launch(q, q_stride, out, out_stride, kcache, vcache, block_tables, bt_stride, tiles, n_tiles, nh,
                                          nkvh, dh, page_shift, scale, window, stream);
    if (q_stride % 8 || out_stride % 4 || ((uintptr_t)q & 15) || ((uintptr_t)out & 7) ||
        ((uintptr_t)kcache & 15) || ((uintptr_t)vcache & 15) || ((uintptr_t)tiles & 15)) return IC_ERR_ARG;
    if (parts < 1) parts = 1;
    if (parts > 1) {
        if (groups == 2 || part_len < 1 || parts > 64 || (long long)nh * n_tiles > kPfCounters || !scratch || !counters ||
            ((uintptr_t)scratch & 15) || scratch_floats < ic_attn_prefill_scratch_floats(n_tiles, nh, dh, parts) ||
            (long long)nh * n_tiles * parts > 0x7fffffffLL) return IC_ERR_ARG;
        groups = 1;
    }
    const float sl2 = scale * 1.4426950408889634f;
    const bool staged = bt_stride <= kPfMaxPages;       // a block never needs more page ids than a request has
    // Few blocks (up to 2 per compute unit; measured with 16..64 heads of 64 and 32..40 of 128 over 512..4,096
    // tokens: two groups win up to 2.0 blocks a unit by 5..25 %, one group from 2.25 on by 2..25 %): the longest
    // tile's walk over the keys sets the time, so two wave groups share it.  Many blocks: one group, more blocks resident.
    const bool two_groups = groups ? groups == 2 : (long long)nh * n_tiles <= 2LL * compute_units();
    dim3 grid((unsigned)nh * (unsigned)n_tiles * (unsigned)parts);
    const bool page64 = page_size >= kPfKeys;            // (a power of two) a 64-key tile lies in one page
#define IC_PF_LAUNCH(DD, ST, GG, PP)                                                                                   \
    hipLaunchKernelGGL((attn_prefill_mfma_kernel<DD, ST, GG, PP>), grid, dim3(256 * GG), 0, stream, (const uint16_t*)q, \
                       q_stride, (uint16_t*)out, out_stride, (const uint16_t*)kcache, (const uint16_t*)vcache,      \
                       block_tables, bt_stride, (const int4*)tiles, n_tiles, nh, nkvh, page_shift, sl2, window,      \
                       parts, part_len, scratch, counters)
#define IC_PF_GROUPS(DD, ST) do { if (two_groups) { if (page64) IC_PF_LAUNCH(DD, ST, 2, true); else IC_PF_LAUNCH(DD, ST, 2, false); } \
                                  else { if (page64) IC_PF_LAUNCH(DD, ST, 1, true); else IC_PF_LAUNCH(DD, ST, 1, false); } } while (0)
    if (dh == 64) { if (staged) IC_PF_GROUPS(64, true); else IC_PF_GROUPS(64, false); }
    else if (dh == 128) { if (staged) IC_PF_GROUPS(128, true); else IC_PF_GROUPS(128, false); }
#undef IC_PF_GROUPS
#undef IC_PF_LAUNCH
    else
        return IC_ERR_UNSUPPORTED;
    return ic_launch_status();
}

IC_EXPORT int ic_attn_prefill_groups(const void* q, int q_stride, void* out, int out_stride, int dtype,
                                     const void* kcache, const void* vcache, const int* block_tables,
                                     int bt_stride, const int* tiles, int n_tiles, int nh, int nkvh, int dh,
                                     int page_size, float scale, int window, int groups, hipStream_t stream) {
    return ic_attn_prefill_split(q, q_stride, out, out_stride, dtype, kcache, vcache, block_tables, bt_stride, tiles,
                                 n_tiles, nh, nkvh, dh, page_size, scale, window, groups, 1, 0, nullptr, 0, nullptr, stream);
}

IC_EXPORT int ic_attn_prefill(const void* q, int q_stride, void* out, int out_stride, int dtype,
                              const void* kcache, const void* vcache, const int* block_tables,
                              int bt_stride, const int* tiles, int n_tiles, int nh, int nkvh, int dh,
                              int page_size, float scale, int window, hipStream_t stream) {
    return ic_attn_prefill_groups(q, q_stride, out, out_stride, dtype, kcache, vcache, block_tables, bt_stride, tiles,
                                  n_tiles, nh, nkvh, dh, page_size, scale, window, 0, stream);
}
