// Attention of single new tokens over the paged cache (decoding), split over
// the keys so that few requests still fill the chip.
//
// Pass 1, grid (splits, kv heads, tokens), 256 threads: a block streams its
// share of one request's keys and values of one kv head once and serves the
// query heads of that group, four at a time.  DH/VEC lanes share a key
// (VEC = 16 bytes of elements per lane), so a wave reads whole contiguous
// rows; every lane keeps a float32 running softmax for its keys, which are
// merged across the lane groups, the four waves, and (pass 2) the splits.
// Pass 2, grid (tokens * heads): combines the splits and writes the output.
//
// Cache layout of one layer: K and V planes [num_pages, n_kv_heads, page_size, head_dim].
#include "attn_decode_blocks.h"
#include "infinicore_infer_variants.h"

template <typename T, int DH, int GQ, bool STAGED>
__global__ void __launch_bounds__(kDecThreads)
attn_decode_split_kernel(const T* __restrict__ q, int q_stride,
                         const T* __restrict__ kcache, const T* __restrict__ vcache,
                         const int* __restrict__ block_tables, int bt_stride,
                         const int* __restrict__ tok_list, const int* __restrict__ token_req,
                         const int* __restrict__ positions,
                         float* __restrict__ part_acc, float* __restrict__ part_ml,
                         int nh, int nkvh, int page_size, float scale, int window, int nsplit, PageDivider div,
                         T* __restrict__ final_out, int out_stride) {
    __shared__ float sm_acc[kDecWaves][GQ][DH];
    __shared__ float sm_ml[kDecWaves][GQ][2];
    __shared__ int pages[kDecMaxPages];
    split_block<T, DH, GQ, STAGED>(q, q_stride, kcache, vcache, block_tables, bt_stride, tok_list, token_req, positions, part_acc, part_ml, nh, nkvh,
                                   page_size, scale, window, nsplit, div, final_out, out_stride, blockIdx.x, blockIdx.y, blockIdx.z, sm_acc, sm_ml, pages);
}

// Grid (tokens * heads), four waves.  Lane s of every wave holds split s (at most 64 splits): the
// weights exp(m_s - max) come from one wave reduction, which every wave does for itself (through LDS: a barrier, 0.1..0.2 us).  Thread (d, g) sums output dim d over
// the splits g, g + G, .. (G = 256 / DH groups, CNT = ceil(splits / G) of them a thread), and the
// groups meet in LDS: with many splits (few kv heads, few requests) one wave alone would walk them
// one after the other.  The partial sums are loaded first, without condition (a slot beyond the
// splits reads the last split and is not added): they do not wait for the weights, so the kernel
// is one round trip to memory, not two.
constexpr int kRedThreads = 256;
template <typename T, int DH, int CNT>
__global__ void __launch_bounds__(kRedThreads)
attn_decode_reduce_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml,
                          const int* __restrict__ tok_list, T* __restrict__ out,
                          int out_stride, int nh, int nsplit) {
    constexpr int G = kRedThreads / DH;
    static_assert(kRedThreads % DH == 0, "every thread has a (dim, group) place");
    __shared__ float grp[kRedThreads];
    const int n = blockIdx.x / nh, h = blockIdx.x % nh, tid = threadIdx.x, lane = tid & 63;
    const size_t base = ((size_t)n * nh + h) * nsplit;
    const int g = __builtin_amdgcn_readfirstlane(tid / DH), d = tid - g * DH;     // (a wave is of one group)
    float pa[CNT];
#pragma unroll
    for (int i = 0; i < CNT; ++i) {
        const int s = (g + i * G < nsplit) ? g + i * G : nsplit - 1;
        pa[i] = part_acc[(base + s) * DH + d];
    }
    const int ls_i = (lane < nsplit) ? lane : nsplit - 1;
    float ms = part_ml[(base + ls_i) * 2], ls = part_ml[(base + ls_i) * 2 + 1];
    const int t = tok_list ? tok_list[n] : n;
    if (lane >= nsplit) { ms = -INFINITY; ls = 0.f; }
    const float mm = wave_max(ms);
    const float w = (ms == -INFINITY) ? 0.f : expf(ms - mm);
    const float inv = 1.0f / wave_sum_of_products(ls, w);
    float a = 0.f;
#pragma unroll
    for (int i = 0; i < CNT; ++i)
        if (g + i * G < nsplit) a += pa[i] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), g + i * G));
    grp[tid] = a;
    __syncthreads();
    if (tid < DH) {
#pragma unroll
        for (int j = 1; j < G; ++j) a += grp[j * DH + tid];
        out[(size_t)t * out_stride + (size_t)h * DH + tid] = from_f32<T>(a * inv);
    }
}

// Grouped queries on the matrix cores: attn_decode_blocks.h.
template <int DH, bool STAGED, int WV>
__global__ void __launch_bounds__(64 * WV, 2)
attn_decode_gqa_kernel(const uint16_t* __restrict__ q, int q_stride,
                       const uint16_t* __restrict__ kcache, const uint16_t* __restrict__ vcache,
                       const int* __restrict__ block_tables, int bt_stride,
                       const int* __restrict__ tok_list, const int* __restrict__ token_req,
                       const int* __restrict__ positions,
                       float* __restrict__ part_acc, float* __restrict__ part_ml,
                       int nh, int nkvh, int page_size, float scale, int window, int nsplit, PageDivider div,
                       uint16_t* __restrict__ final_out, int out_stride) {
    __shared__ __attribute__((aligned(16))) uint16_t Vs[gqa_tile_elements<DH, WV>()];
    __shared__ float sm_ml[WV][16][2];
    __shared__ int pages[kDecMaxPages];
    gqa_block<DH, STAGED, WV>(q, q_stride, kcache, vcache, block_tables, bt_stride, tok_list, token_req, positions, part_acc, part_ml, nh, nkvh,
                              page_size, scale, window, nsplit, div, final_out, out_stride, blockIdx.x, blockIdx.y, blockIdx.z, Vs, sm_ml, pages);
}

// Grouped queries in bfloat16 run the matrix-core kernel: the one place that says so (the key-split rule asks here too).
IC_EXPORT int ic_attn_decode_on_matrix_cores(int dtype, int n_heads, int n_kv_heads) { return dtype == IC_BF16 && n_heads != n_kv_heads; }

IC_EXPORT int ic_attn_decode_page_of(int key, int page_size) { return key < 0 || page_size <= 0 ? -1 : PageDivider(page_size).page_of(key); }

// Waves of a block of the grouped-query kernel: eight where one split's share is long for four and the blocks are too few to fill the units anyway
// (24:8 heads of 64, one split: 258 keys 5.4 -> 5.1 us, 16 rows of up to 2,000 keys 17.7 -> 13.7; with 320 pairs of 1,000 keys 18.7 -> 20.5).
// Heads of 128 and shares of several splits gain little by them (32:2 heads, 16,385 keys in 32 splits 22.5 -> 21.3, 500 keys in one 12.6 -> 12.2; 24:8
// heads of 64, 4,000 keys in 32 splits 8.2 -> 8.6).
IC_EXPORT int ic_attn_decode_waves(int head_dim, int pairs, int nsplit) { return head_dim == 64 && nsplit == 1 && pairs <= 128 ? 8 : kDecWaves; }

// The second pass: sums the splits' results.
template <typename T, int DH>
static int launch_merge(const float* part_acc, const float* part_ml, const int* tok_list, void* out, int out_stride, int n_tok, int nh, int nsplit,
                        hipStream_t stream) {
    const int per_thread = (nsplit + kRedThreads / DH - 1) / (kRedThreads / DH);    // splits a thread of the second pass sums
#define IC_RED_LAUNCH(CNT)                                                                                      \
    hipLaunchKernelGGL((attn_decode_reduce_kernel<T, DH, CNT>), dim3(n_tok * nh), dim3(kRedThreads), 0, stream, \
                       part_acc, part_ml, tok_list, (T*)out, out_stride, nh, nsplit)
    if (per_thread <= 2) IC_RED_LAUNCH(2);
    else if (per_thread <= 4) IC_RED_LAUNCH(4);
    else if (per_thread <= 8) IC_RED_LAUNCH(8);
    else if (per_thread <= 16) IC_RED_LAUNCH(16);
    else IC_RED_LAUNCH(32);                             // 64 splits, two groups
#undef IC_RED_LAUNCH
    return ic_launch_status();
}

template <typename T, int DH>
static int launch_decode(const void* q, int q_stride, void* out, int out_stride, const void* kcache,
                         const void* vcache, const int* block_tables, int bt_stride, const int* tok_list,
                         const int* token_req, const int* positions, float* part_acc, float* part_ml,
                         int n_tok, int nh, int nkvh, int page_size, float scale, int window, int nsplit,
                         hipStream_t stream) {
    dim3 grid(nsplit, nkvh, n_tok), block(kDecThreads);
    const bool staged = bt_stride <= kDecMaxPages;      // a block never needs more page ids than a request has
    const PageDivider div(page_size);
    void* direct = (nsplit == 1) ? out : nullptr;       // one split writes the result itself
#define IC_DEC_LAUNCH(KERNEL, TQ)                                                                           \
    hipLaunchKernelGGL(KERNEL, grid, block, 0, stream, (const TQ*)q, q_stride, (const TQ*)kcache,           \
                       (const TQ*)vcache, block_tables, bt_stride, tok_list, token_req, positions, part_acc, \
                       part_ml, nh, nkvh, page_size, scale, window, nsplit, div, (TQ*)direct, out_stride)
    if (ic_attn_decode_on_matrix_cores(sizeof(T) == 2 ? IC_BF16 : IC_F32, nh, nkvh)) {
        const bool eight = ic_attn_decode_waves(DH, n_tok * nkvh, nsplit) == 8;
        if constexpr (DH == 64) {
            if (eight) {
                block = dim3(512);
                if (staged) IC_DEC_LAUNCH((attn_decode_gqa_kernel<DH, true, 8>), uint16_t);
                else IC_DEC_LAUNCH((attn_decode_gqa_kernel<DH, false, 8>), uint16_t);
            }
        }
        if (eight) { /* launched */ }
        else if (staged) IC_DEC_LAUNCH((attn_decode_gqa_kernel<DH, true, 4>), uint16_t);
        else IC_DEC_LAUNCH((attn_decode_gqa_kernel<DH, false, 4>), uint16_t);
    } else if (nh == nkvh) {
        if (staged) IC_DEC_LAUNCH((attn_decode_split_kernel<T, DH, 1, true>), T);
        else IC_DEC_LAUNCH((attn_decode_split_kernel<T, DH, 1, false>), T);
    } else {
        if (staged) IC_DEC_LAUNCH((attn_decode_split_kernel<T, DH, 4, true>), T);
        else IC_DEC_LAUNCH((attn_decode_split_kernel<T, DH, 4, false>), T);
    }
#undef IC_DEC_LAUNCH
    int st = ic_launch_status();
    if (st || nsplit == 1) return st;
    return launch_merge<T, DH>(part_acc, part_ml, tok_list, out, out_stride, n_tok, nh, nsplit, stream);
}

// Head sizes with a tiled decode kernel.
IC_EXPORT int ic_attn_decode_supported(int dtype, int dh) {
    return (dtype == IC_F32 || dtype == IC_BF16) && (dh == 64 || dh == 128);
}

// order[r] = the row whose position is the r-th largest (of equal ones the first): where more blocks are launched than the chip holds
// at once, the longest walks over the keys must not be the last to start.  One block; n rows at most kOrderRows.
constexpr int kOrderRows = 1024;
__global__ void __launch_bounds__(kOrderRows)
attn_decode_order_kernel(const int* __restrict__ positions, int* __restrict__ order, int n) {
    __shared__ int pos[kOrderRows];
    const int i = threadIdx.x;
    const int mine = i < n ? positions[i] : 0;
    pos[i] = mine;
    __syncthreads();
    if (i >= n) return;
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += (pos[j] > mine || (pos[j] == mine && j < i)) ? 1 : 0;
    order[rank] = i;
}

// Whether a step of n_rows single tokens, all its rows, is worth the kernel above (once a step 1.8 us for 8 rows, 2.9 for 64, 38 for 1,000): 64 rows of 36
// heads of 64 over 300..2,100 keys 95.0 -> 88.8 us a layer, 40 rows of 24:8 heads over 100..2,048 22.3 -> 20.4, 24 rows of 36 heads over 100..1,500 27.5 ->
// 26.1, 9 over 100..1,000 14.6 -> 11.7.  Rows of one length gain nothing and pay for it (the step may be a recorded one, whose lengths the host does not
// know).  Several splits balance the walks already (16 rows of 36 heads in 4 splits 27.0 and 28.4), and up to one block a unit all start at once.
IC_EXPORT int ic_attn_decode_wants_order(int n_rows, int nkvh, int nsplit, int compute_units) {
    return nsplit == 1 && n_rows > 1 && n_rows <= kOrderRows && (long long)n_rows * nkvh > (compute_units > 0 ? compute_units : 256);
}

IC_EXPORT int ic_attn_decode_order(const int* positions, int* order, int n_rows, hipStream_t stream) {
    if (n_rows <= 0) return IC_OK;
    if (n_rows > kOrderRows || !positions || !order) return IC_ERR_ARG;
    hipLaunchKernelGGL(attn_decode_order_kernel, dim3(1), dim3((n_rows + 63) / 64 * 64), 0, stream, positions, order, n_rows);
    return ic_launch_status();
}

IC_EXPORT int ic_attn_decode_merge(const float* part_acc, const float* part_ml, const int* tok_list, void* out, int out_stride, int dtype, int n_tok, int nh,
                                   int dh, int nsplit, hipStream_t stream) {
    if (n_tok <= 0) return IC_OK;
    if (!part_acc || !part_ml || !out || nh <= 0 || nsplit <= 0 || nsplit > 64 || dtype != IC_BF16) return IC_ERR_ARG;
    if (dh == 64) return launch_merge<bf16, 64>(part_acc, part_ml, tok_list, out, out_stride, n_tok, nh, nsplit, stream);
    if (dh == 128) return launch_merge<bf16, 128>(part_acc, part_ml, tok_list, out, out_stride, n_tok, nh, nsplit, stream);
    return IC_ERR_UNSUPPORTED;
}

// part_acc: float32 [n_tok, nh, nsplit, dh]; part_ml: float32 [n_tok, nh, nsplit, 2].
// tok_list: rows of q/out that are decoded (nullptr: rows 0..n_tok-1).
IC_EXPORT int ic_attn_decode(const void* q, int q_stride, void* out, int out_stride, int dtype,
                             const void* kcache, const void* vcache, const int* block_tables,
                             int bt_stride, const int* tok_list, const int* token_req,
                             const int* positions, float* part_acc, float* part_ml, int n_tok, int nh,
                             int nkvh, int dh, int page_size, float scale, int window, int nsplit,
                             hipStream_t stream) {
    if (n_tok <= 0) return IC_OK;
    if (nh <= 0 || nkvh <= 0 || nh % nkvh || page_size <= 0 || nsplit <= 0 || nsplit > 64) return IC_ERR_ARG;
    if (nkvh > 65535 || n_tok > 65535) return IC_ERR_ARG;
    if (q_stride % 8 || ((uintptr_t)q & 15) || ((uintptr_t)kcache & 15) || ((uintptr_t)vcache & 15)) return IC_ERR_ARG;
#define IC_DECODE_CASE(TT, DD)                                                                          \
    return launch_decode<TT, DD>(q, q_stride, out, out_stride, kcache, vcache, block_tables, bt_stride, \
                                 tok_list, token_req, positions, part_acc, part_ml, n_tok, nh, nkvh,   \
                                 page_size, scale, window, nsplit, stream)
    if (dtype == IC_F32 && dh == 64) IC_DECODE_CASE(float, 64);
    if (dtype == IC_F32 && dh == 128) IC_DECODE_CASE(float, 128);
    if (dtype == IC_BF16 && dh == 64) IC_DECODE_CASE(bf16, 64);
    if (dtype == IC_BF16 && dh == 128) IC_DECODE_CASE(bf16, 128);
#undef IC_DECODE_CASE
    return IC_ERR_UNSUPPORTED;
}
