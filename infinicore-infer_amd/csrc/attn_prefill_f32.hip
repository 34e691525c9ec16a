// Attention of prompt portions over the paged cache in true float32 on the matrix cores
// (v_mfma_f32_32x32x2_f32: float32 operands, float32 accumulation, no reduced-precision mode).
//
// The 32-bit path's prompts otherwise run in the general kernel, one wave per (token, head) with scalar
// dot products: 3.5 ms a layer for a 2,048-token prompt of the 2B shape, two thirds of that path's prompt
// time.  Here a block of four waves owns up to 128 consecutive tokens of one request and one head, wave w
// rows 32 w .. 32 w + 31, and walks the keys 64 at a time through LDS, as the bfloat16 kernel does; the
// tile list is the same.  Scores are computed transposed, S^T = K Q^T, so a lane holds 32 keys of ONE query
// and the running softmax needs a single cross-lane step; the probabilities are then already the B operand
// of O^T = V^T P^T.
//
// 32x32x2 operand layout (lane l, h = l / 32): A[i = l % 32][k = h], B[k = h][j = l % 32],
// D[i = 8 (r / 4) + 4 h + r % 4][j = l % 32] for the 16 accumulators r.  Which two values of the summed
// dimension an instruction takes is free as long as A and B agree: in S^T = K Q^T instruction c takes head
// dims c and c + DH / 2 (so a lane's K operands are DH / 2 consecutive floats of its key's row), and in
// O^T = V^T P^T accumulator r of S^T is the B operand as it stands: it holds key 8 (r / 4) + r % 4 in the
// lower half of the wave and the key four further on in the upper half.
//
// The float32 matrix instructions take 16 times as long as the bfloat16 ones, so what counts is that every SIMD has some: with
// few tiles (a portion of 512 tokens of 24 heads makes 96) a block of four waves takes only 64 or 32 of a tile's rows and its waves
// share the keys between them, KG key groups of 32 keys a step, merged through LDS at the end.  The next step's keys and
// values are on their way in registers while this one's are used.
//
// Cache layout of one layer: K and V planes [num_pages, n_kv_heads, page_size, head_dim].
#include "common.h"

typedef float f32_v16 __attribute__((ext_vector_type(16)));

constexpr int kF32Threads = 256;
constexpr int kF32Rows = 128;     // query rows per block (must equal the bfloat16 kernel's tile height: one tile list serves both)

// KG key groups: 1 (a step of 64 keys, every wave all of them), 2 (64 keys, 32 a group) or 4 (128 keys, 32 a group).
template <int DH, int KG>
__global__ void __launch_bounds__(kF32Threads, (KG == 4 || DH == 128) ? 1 : 2)
attn_prefill_f32_kernel(const float* __restrict__ q, int q_stride, float* __restrict__ out, int out_stride,
                        const float* __restrict__ kcache, const float* __restrict__ vcache,
                        const int* __restrict__ block_tables, int bt_stride, const int4* __restrict__ tiles,
                        int n_tiles, int nh, int nkvh, int page_shift, float scale_log2e, int window) {
    constexpr int HALF = DH / 2;          // matrix instructions per 32-key tile of S^T
    constexpr int ND = DH / 32;           // 32-row tiles of O^T
    constexpr int KS = DH + 4;            // row stride of the K tile (floats): 16-byte reads of 16 consecutive rows cover all banks
    constexpr int VS = DH + 8;            // row stride of the V tile: rows four apart (the wave's two halves) fall into different banks
    constexpr int KEYS = KG == 4 ? 128 : 64;                  // keys per step
    constexpr int GK = KG == 1 ? 64 : 32;                     // of them, a group's
    constexpr int NT = GK / 32;                               // 32-key tiles of a group
    constexpr int RW = 4 / KG;                                // waves that own rows, 32 each
    constexpr int NL = KEYS * (DH / 4) / kF32Threads;         // 16-byte loads per thread and plane
    constexpr int MF = 2 + ND * 16;                           // floats a lane hands over at the end
    static_assert(KG == 1 || KEYS * (KS + VS) >= (4 - RW) * 64 * MF, "the merge buffer fits in the tiles");
    __shared__ __attribute__((aligned(16))) float tile_mem[KEYS * (KS + VS)];
    float* const Ks = tile_mem;
    float* const Vs = tile_mem + KEYS * KS;

    const int slot = (int)blockIdx.x / KG, sub = (int)blockIdx.x % KG;      // tile-major: all heads of the longest tile first
    const int h = slot % nh;
    const int4 tile = tiles[slot / nh];
    const int skip = 32 * RW * sub;                           // rows of the tile before this block's
    const int req = tile.x, row0 = tile.y + skip, pos0 = tile.w + skip;
    const int n_rows = tile.z - skip < 32 * RW ? tile.z - skip : 32 * RW;
    if (n_rows <= 0) return;                                  // (the whole block)
    const int kvh = h / (nh / nkvh);
    const int* bt = block_tables + (size_t)req * bt_stride;
    const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) % RW, grp = (tid >> 6) / RW;
    const int lq = lane & 31, half = lane >> 5;
    const int page_size = 1 << page_shift, page_mask = page_size - 1;

    const int my_row = 32 * wave + lq;
    const bool row_ok = my_row < n_rows;
    const int qpos = pos0 + my_row;
    const bool wave_ok = 32 * wave < n_rows;
    const int wave_first = pos0 + 32 * wave;
    const int wave_last = pos0 + ((32 * wave + 31 < n_rows - 1) ? 32 * wave + 31 : n_rows - 1);
    const int last_key = pos0 + n_rows - 1;
    int first_key = 0;
    if (window > 0 && pos0 - window + 1 > 0) first_key = pos0 - window + 1;
    const int kb_begin = (first_key / KEYS) * KEYS;

    // Q operands: Q[query lq][HALF * half + c], scores in units of log 2 (the softmax scale folded in)
    float qf[HALF];
    {
        const float* qp = q + (size_t)(row0 + (row_ok ? my_row : 0)) * q_stride + (size_t)h * DH + HALF * half;
#pragma unroll
        for (int c = 0; c < HALF; c += 4) {
            const float4 v = *reinterpret_cast<const float4*>(qp + c);
            qf[c] = row_ok ? v.x * scale_log2e : 0.f; qf[c + 1] = row_ok ? v.y * scale_log2e : 0.f;
            qf[c + 2] = row_ok ? v.z * scale_log2e : 0.f; qf[c + 3] = row_ok ? v.w * scale_log2e : 0.f;
        }
    }
    f32_v16 oacc[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
    float m = -INFINITY, l = 0.f;

    const size_t head_stride = (size_t)page_size * DH;
    const float* kbase = kcache + (size_t)kvh * head_stride;
    const float* vbase = vcache + (size_t)kvh * head_stride;
    const size_t page_stride = (size_t)nkvh * head_stride;

    // a step's keys and values (those outside the tile's range as zeros: they are masked)
    float4 kr[NL], vr[NL];
    auto fetch = [&](int kb) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int idx = tid + i * kF32Threads;
            const int key = idx / (DH / 4), quad = idx - key * (DH / 4);
            const int ka = kb + key;
            kr[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            vr[i] = kr[i];
            if (ka <= last_key && ka >= first_key) {
                const size_t off = (size_t)bt[ka >> page_shift] * page_stride + (size_t)(ka & page_mask) * DH + quad * 4;
                kr[i] = *reinterpret_cast<const float4*>(kbase + off);
                vr[i] = *reinterpret_cast<const float4*>(vbase + off);
            }
        }
    };
    fetch(kb_begin);
    for (int kb = kb_begin; kb <= last_key; kb += KEYS) {
        __syncthreads();                                // the previous step's readers are done
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int idx = tid + i * kF32Threads;
            const int key = idx / (DH / 4), quad = idx - key * (DH / 4);
            *reinterpret_cast<float4*>(&Ks[key * KS + quad * 4]) = kr[i];
            *reinterpret_cast<float4*>(&Vs[key * VS + quad * 4]) = vr[i];
        }
        __syncthreads();
        if (kb + KEYS <= last_key) fetch(kb + KEYS);    // in flight while this step is used
        const int kt = kb + GK * grp;                   // this group's keys
        if (!wave_ok || kt > wave_last) continue;       // nothing this wave may see
        if (window > 0 && kt + GK - 1 < wave_first - window + 1) continue;
        const float* const Kg = Ks + GK * grp * KS;
        const float* const Vg = Vs + GK * grp * VS;

        // ---- S^T = K Q^T : tiles of 32 keys ----------------------------------------------------------
        f32_v16 sacc[NT];
#pragma unroll
        for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sacc[tt][r] = 0.f;
            const float* kp = &Kg[(32 * tt + lq) * KS + HALF * half];
#pragma unroll
            for (int c = 0; c < HALF; c += 4) {
                const float4 kx = *reinterpret_cast<const float4*>(kp + c);
                sacc[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx.x, qf[c], sacc[tt], 0, 0, 0);
                sacc[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx.y, qf[c + 1], sacc[tt], 0, 0, 0);
                sacc[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx.z, qf[c + 2], sacc[tt], 0, 0, 0);
                sacc[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx.w, qf[c + 3], sacc[tt], 0, 0, 0);
            }
        }
        // ---- mask (only steps that touch the diagonal, the window's edge, or keys before the window) --------
        const bool need_mask = (kt + GK - 1 > wave_first) || (window > 0);
        if (need_mask) {
            // key kt + 4 half + e of this lane's accumulator (e a constant per accumulator) is seen when e <= lim
            const int lim = qpos - kt - 4 * half;
#pragma unroll
            for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (32 * tt + 8 * (r >> 2) + (r & 3) > lim) sacc[tt][r] = -INFINITY;
            if (window > 0) {
#pragma unroll
                for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (32 * tt + 8 * (r >> 2) + (r & 3) <= lim - window) sacc[tt][r] = -INFINITY;
            }
        }
        // ---- running softmax, base 2 -------------------------------------------------------------------
        float mloc = sacc[0][0];
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
            for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, sacc[tt][r]);
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32, kWave));
        const float m_new = fmaxf(m, mloc);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float corr = exp2f(m - m_use);            // 0 on the first step (m = -inf)
        float rs = 0.f;
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float p = exp2f(sacc[tt][r] - m_use);
                sacc[tt][r] = p;
                rs += p;
            }
        rs += __shfl_xor(rs, 32, kWave);
        l = l * corr + rs;
        m = m_new;
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] *= corr;

        // ---- O^T += V^T P^T : accumulator r of S^T is the B operand as it stands -------------------------------
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float* vp = &Vg[(32 * tt + 8 * (r >> 2) + 4 * half + (r & 3)) * VS + lq];
#pragma unroll
                for (int dt = 0; dt < ND; ++dt)
                    oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vp[32 * dt], sacc[tt][r], oacc[dt], 0, 0, 0);
            }
    }

    // ---- the key groups' states meet in group 0 (same lane, same rows) ---------------------------------------
    if constexpr (KG > 1) {
        __syncthreads();                                // the last step's readers are done
        float* const mine = tile_mem + (size_t)((grp > 0 ? grp - 1 : 0) * RW + wave) * 64 * MF + lane;
        if (grp > 0) {
            mine[0] = m;
            mine[64] = l;
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) mine[(2 + 16 * i + r) * 64] = oacc[i][r];
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 0; g < KG - 1; ++g) {
            const float* const other = tile_mem + (size_t)(g * RW + wave) * 64 * MF + lane;
            const float m1 = other[0], l1 = other[64];
            const float m_new = fmaxf(m, m1);
            const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
            const float c0 = exp2f(m - m_use), c1 = exp2f(m1 - m_use);
            l = l * c0 + l1 * c1;
            m = m_new;
#pragma unroll
            for (int i = 0; i < ND; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[i][r] = oacc[i][r] * c0 + other[(2 + 16 * i + r) * 64] * c1;
        }
    }
    if (!row_ok) return;
    const float inv = 1.0f / l;
    float* op = out + (size_t)(row0 + my_row) * out_stride + (size_t)h * DH;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
            const int d = 32 * dt + 8 * rg + 4 * half;
            *reinterpret_cast<float4*>(op + d) = make_float4(oacc[dt][4 * rg] * inv, oacc[dt][4 * rg + 1] * inv,
                                                             oacc[dt][4 * rg + 2] * inv, oacc[dt][4 * rg + 3] * inv);
        }
}

// Called by ic_attn_prefill_split for float32 (attn_prefill_mfma.hip): the arguments are checked there.
int ic_attn_prefill_f32_launch(const void* q, int q_stride, void* out, int out_stride, const void* kcache, const void* vcache,
                               const int* block_tables, int bt_stride, const int* tiles, int n_tiles, int nh, int nkvh, int dh,
                               int page_shift, float scale, int window, hipStream_t stream) {
    if (q_stride % 4 || out_stride % 4 || ((uintptr_t)q & 15) || ((uintptr_t)out & 15) || ((uintptr_t)kcache & 15) ||
        ((uintptr_t)vcache & 15) || ((uintptr_t)tiles & 15))
        return IC_ERR_ARG;
    const float sl2 = scale * 1.4426950408889634f;
    // Key groups from the number of (tile, head) pairs; one / two / four groups, us (24:8, 36:36 heads of 64; 32:2 of 128): 96 pairs (509
    // tokens after 130; the kernel without groups and loads ahead took 70) 58 / 38 / 35; 144 (512 tokens) 47 / 35 / 33; 192 (window of
    // 300) 45 / 39 / 53; 288 (1,024 tokens) 100 / 78 / 88; 576 (2,048) 248 / 230 / 280; of 128: 96 (300 after 1,000) 215 / 138 / 162;
    // 128 (512) 86 / 58 / 54; 384 (1,500) 268 / 295 / 356.
    const long long pairs = (long long)nh * n_tiles;
    const int kg = dh == 64 ? (pairs <= 160 ? 4 : pairs <= 700 ? 2 : 1) : (pairs <= 256 ? 2 : 1);
    if (pairs * kg > 0x7fffffffLL) return IC_ERR_ARG;
    dim3 grid((unsigned)nh * (unsigned)n_tiles * (unsigned)kg), block(kF32Threads);
#define IC_F32_LAUNCH(DD, GG)                                                                                            \
    hipLaunchKernelGGL((attn_prefill_f32_kernel<DD, GG>), grid, block, 0, stream, (const float*)q, q_stride, (float*)out, \
                       out_stride, (const float*)kcache, (const float*)vcache, block_tables, bt_stride,                  \
                       (const int4*)tiles, n_tiles, nh, nkvh, page_shift, sl2, window)
    if (dh == 64) { if (kg == 1) IC_F32_LAUNCH(64, 1); else if (kg == 2) IC_F32_LAUNCH(64, 2); else IC_F32_LAUNCH(64, 4); }
    else if (dh == 128) { if (kg == 1) IC_F32_LAUNCH(128, 1); else IC_F32_LAUNCH(128, 2); }
    else return IC_ERR_UNSUPPORTED;
#undef IC_F32_LAUNCH
    return ic_launch_status();
}
