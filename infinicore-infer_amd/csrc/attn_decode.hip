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
#include "common.h"

constexpr int kDecThreads = 256;
constexpr int kDecWaves = kDecThreads / 64;
constexpr int kDecUnroll = 4;
constexpr int kDecMaxPages = 1024;   // page ids of one block's keys staged in LDS (else read from memory)

template <typename T> struct Vec16;
template <> struct Vec16<float> {
    static constexpr int N = 4;
    __device__ static uint4 raw(const float* p) { return load_stream16(p); }
    __device__ static void unpack(const uint4& v, float* o) {
        o[0] = __uint_as_float(v.x); o[1] = __uint_as_float(v.y);
        o[2] = __uint_as_float(v.z); o[3] = __uint_as_float(v.w);
    }
    __device__ static void load(const float* p, float* o) { unpack(raw(p), o); }
};
template <> struct Vec16<bf16> {
    static constexpr int N = 8;
    __device__ static uint4 raw(const bf16* p) { return load_stream16(p); }
    __device__ static void unpack(const uint4& v, float* o) {
        o[0] = __uint_as_float(v.x << 16); o[1] = __uint_as_float(v.x & 0xffff0000u);
        o[2] = __uint_as_float(v.y << 16); o[3] = __uint_as_float(v.y & 0xffff0000u);
        o[4] = __uint_as_float(v.z << 16); o[5] = __uint_as_float(v.z & 0xffff0000u);
        o[6] = __uint_as_float(v.w << 16); o[7] = __uint_as_float(v.w & 0xffff0000u);
    }
    __device__ static void load(const bf16* p, float* o) { unpack(raw(p), o); }
};

// merge running-softmax state b into a
__device__ __forceinline__ void merge_state(float& m, float& l, float* acc, int n,
                                            float mb, float lb, const float* accb) {
    const float mn = fmaxf(m, mb);
    if (mn == -INFINITY) return;                 // both empty
    const float ca = __builtin_amdgcn_exp2f(m - mn), cb = __builtin_amdgcn_exp2f(mb - mn);   // maxima in units of log 2
    l = l * ca + lb * cb;
    for (int i = 0; i < n; ++i) acc[i] = acc[i] * ca + accb[i] * cb;
    m = mn;
}

template <typename T, int DH, int GQ, bool STAGED>
__global__ void __launch_bounds__(kDecThreads)
attn_decode_split_kernel(const T* __restrict__ q, int q_stride,
                         const T* __restrict__ kcache, const T* __restrict__ vcache,
                         const int* __restrict__ block_tables, int bt_stride,
                         const int* __restrict__ tok_list, const int* __restrict__ token_req,
                         const int* __restrict__ positions,
                         float* __restrict__ part_acc, float* __restrict__ part_ml,
                         int nh, int nkvh, int page_size, float scale, int window, int nsplit, unsigned page_rcp,
                         T* __restrict__ final_out, int out_stride) {
    constexpr int VEC = Vec16<T>::N;
    constexpr int LPK = DH / VEC;                 // lanes per key
    constexpr int KPW = 64 / LPK;                 // keys per wave per step
    constexpr int KPB = KPW * kDecWaves;          // keys per block per step
    static_assert(DH % VEC == 0 && 64 % LPK == 0, "head size must split a wave evenly");

    __shared__ float sm_acc[kDecWaves][GQ][DH];
    __shared__ float sm_ml[kDecWaves][GQ][2];
    __shared__ int pages[kDecMaxPages];

    const int split = blockIdx.x, kvh = blockIdx.y, n = blockIdx.z;
    const int t = tok_list ? tok_list[n] : n;
    const int g = nh / nkvh;
    const int pos = positions[t];
    const int* bt = block_tables + (size_t)token_req[t] * bt_stride;
    const int lo0 = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    const int nkeys = pos + 1 - lo0;
    const int per = (nkeys + nsplit - 1) / nsplit;
    const int lo = lo0 + split * per;
    int hi = lo + per;
    if (hi > pos + 1) hi = pos + 1;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane % LPK;                   // which 16-byte slice of the row
    const int grp = lane / LPK;                   // which key of the wave's step
    const size_t head_stride = (size_t)page_size * DH;
    const size_t page_stride = (size_t)nkvh * head_stride;
    const T* kbase = kcache + (size_t)kvh * head_stride + sub * VEC;
    const T* vbase = vcache + (size_t)kvh * head_stride + sub * VEC;

    // page ids of this block's keys, staged once: the loop then needs one memory hop per key.
    // STAGED is a compile-time choice (the host knows the block table's width): a run-time choice
    // between the two arrays would make every lookup a flat load, whose wait also waits for the
    // key and value loads in flight.
    // A request whose ids are staged has at most kDecMaxPages pages, so key / page_size is one multiplication by
    // page_rcp = ceil(2^32 / page_size) instead of some 20 instructions.
    auto page_of = [&](int key) { return STAGED ? (int)__umulhi((unsigned)key, page_rcp) : key / page_size; };
    const int page_lo = page_of(lo);
    const int n_pages = (hi > lo) ? page_of(hi - 1) - page_lo + 1 : 0;
    if (STAGED)
        for (int i = threadIdx.x; i < n_pages; i += kDecThreads) pages[i] = bt[page_lo + i];
    __syncthreads();

    // element offset of a key's row piece in a plane
    auto row_of = [&](int key) -> size_t {
        const int lp = page_of(key);
        const int pg = STAGED ? pages[lp - page_lo] : bt[lp];
        return (size_t)pg * page_stride + (size_t)(key - lp * page_size) * DH;
    };

    for (int h0 = 0; h0 < g; h0 += GQ) {
        float qv[GQ][VEC], acc[GQ][VEC], m[GQ], l[GQ];
#pragma unroll
        for (int j = 0; j < GQ; ++j) {
            m[j] = -INFINITY; l[j] = 0.f;
            const int hh = (h0 + j < g) ? h0 + j : g - 1;
            Vec16<T>::load(q + (size_t)t * q_stride + (size_t)(kvh * g + hh) * DH + sub * VEC, qv[j]);
#pragma unroll
            for (int i = 0; i < VEC; ++i) { qv[j][i] *= scale * 1.4426950408889634f; acc[j][i] = 0.f; }   // scores in units of log 2
        }

        // keys kb, kb + KPB, ... of one step; the next step's loads are issued before this one is used
        uint4 kr[2][kDecUnroll], vr[2][kDecUnroll];
        // Loads are unconditional (keys beyond the share read its last key and are ignored), so the
        // loop is straight-line code and a stage waits only for its own loads.
        auto issue = [&](int kb, uint4* kk, uint4* vv) {
#pragma unroll
            for (int u = 0; u < kDecUnroll; ++u) {
                const int key = (kb + u * KPB < hi) ? kb + u * KPB : hi - 1;
                const size_t off = row_of(key);
                kk[u] = Vec16<T>::raw(kbase + off);
                vv[u] = Vec16<T>::raw(vbase + off);
            }
        };
        auto consume = [&](int kb, const uint4* kk, const uint4* vv) {
            float kf[kDecUnroll][VEC];
            bool ok[kDecUnroll];
#pragma unroll
            for (int u = 0; u < kDecUnroll; ++u) {
                ok[u] = kb + u * KPB < hi;
                Vec16<T>::unpack(kk[u], kf[u]);
            }
#pragma unroll
            for (int j = 0; j < GQ; ++j) {
                float s[kDecUnroll];
                float mx = m[j];
#pragma unroll
                for (int u = 0; u < kDecUnroll; ++u) {
                    float d = 0.f;
#pragma unroll
                    for (int i = 0; i < VEC; ++i) d += qv[j][i] * kf[u][i];
                    d = group_sum<LPK>(d);
                    s[u] = ok[u] ? d : -INFINITY;
                    mx = fmaxf(mx, s[u]);
                }
                if (mx == -INFINITY) continue;     // this lane group has seen no key yet
                const float corr = __builtin_amdgcn_exp2f(m[j] - mx);
                float lsum = l[j] * corr;
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc[j][i] *= corr;
#pragma unroll
                for (int u = 0; u < kDecUnroll; ++u) {
                    float vf[VEC];
                    Vec16<T>::unpack(vv[u], vf);
                    const float p = __builtin_amdgcn_exp2f(s[u] - mx);      // 0 for a key beyond the share
                    lsum += p;
#pragma unroll
                    for (int i = 0; i < VEC; ++i) acc[j][i] += p * vf[i];
                }
                l[j] = lsum;
                m[j] = mx;
            }
        };
        constexpr int STEP = kDecUnroll * KPB;
        const int kb0 = lo + wave * KPW + grp;
        if (lo < hi) {                               // (block-uniform) an empty share has no key to read, not even a stand-in
            issue(kb0, kr[0], vr[0]);
            for (int kb = kb0; kb < hi; kb += 2 * STEP) {
                issue(kb + STEP, kr[1], vr[1]);
                consume(kb, kr[0], vr[0]);
                issue(kb + 2 * STEP, kr[0], vr[0]);
                consume(kb + STEP, kr[1], vr[1]);
            }
        }

        // merge the lane groups of the wave (lanes with the same `sub`)
#pragma unroll
        for (int j = 0; j < GQ; ++j) {
#pragma unroll
            for (int o = LPK; o < 64; o <<= 1) {
                const float mb = __shfl_xor(m[j], o, kWave);
                const float lb = __shfl_xor(l[j], o, kWave);
                float ab[VEC];
#pragma unroll
                for (int i = 0; i < VEC; ++i) ab[i] = __shfl_xor(acc[j][i], o, kWave);
                merge_state(m[j], l[j], acc[j], VEC, mb, lb, ab);
            }
        }
        __syncthreads();                            // LDS free from the previous head chunk
        if (grp == 0) {
#pragma unroll
            for (int j = 0; j < GQ; ++j) {
#pragma unroll
                for (int i = 0; i < VEC; ++i) sm_acc[wave][j][sub * VEC + i] = acc[j][i];
                if (sub == 0) { sm_ml[wave][j][0] = m[j]; sm_ml[wave][j][1] = l[j]; }
            }
        }
        __syncthreads();
        // merge the waves: thread (j, d) for j < GQ, d < DH
        for (int idx = threadIdx.x; idx < GQ * DH; idx += kDecThreads) {
            const int j = idx / DH, d = idx - j * DH;
            if (h0 + j >= g) continue;
            float mm = -INFINITY;
            for (int w = 0; w < kDecWaves; ++w) mm = fmaxf(mm, sm_ml[w][j][0]);
            float a = 0.f, ll = 0.f;
            if (mm != -INFINITY) {
                for (int w = 0; w < kDecWaves; ++w) {
                    const float c = __builtin_amdgcn_exp2f(sm_ml[w][j][0] - mm);
                    a += sm_acc[w][j][d] * c;
                    ll += sm_ml[w][j][1] * c;
                }
            }
            const int h = kvh * g + h0 + j;
            if (final_out) {                        // a single split: this is the result, no second pass
                final_out[(size_t)t * out_stride + (size_t)h * DH + d] = from_f32<T>(a / ll);
                continue;
            }
            const size_t pidx = ((size_t)n * nh + h) * nsplit + split;
            part_acc[pidx * DH + d] = a;
            // the partial maximum leaves in natural units, as the second pass expects
            if (d == 0) { part_ml[pidx * 2] = mm * 0.6931471805599453f; part_ml[pidx * 2 + 1] = ll; }
        }
    }
}

// Grid (tokens * heads), four waves.  Lane s of every wave holds split s (at most 64 splits): the
// weights exp(m_s - max) come from one wave reduction.  Thread (d, g) sums output dim d over
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
    __shared__ float wgt[64];
    __shared__ float grp[kRedThreads];
    const int n = blockIdx.x / nh, h = blockIdx.x % nh, tid = threadIdx.x, lane = tid & 63;
    const size_t base = ((size_t)n * nh + h) * nsplit;
    const int g = tid / DH, d = tid - g * DH;
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
    const float inv = 1.0f / wave_sum(ls * w);
    if (tid < 64) wgt[lane] = w;
    __syncthreads();
    float a = 0.f;
#pragma unroll
    for (int i = 0; i < CNT; ++i)
        if (g + i * G < nsplit) a += pa[i] * wgt[g + i * G];
    grp[tid] = a;
    __syncthreads();
    if (tid < DH) {
#pragma unroll
        for (int j = 1; j < G; ++j) a += grp[j * DH + tid];
        out[(size_t)t * out_stride + (size_t)h * DH + tid] = from_f32<T>(a * inv);
    }
}

// ---------------------------------------------------------------------------------------------
// Grouped queries on the matrix cores (bfloat16): the query heads that share a kv head are the
// columns of one 16-wide tile, so keys and values are read once for the whole group.
//
// Same grid and partial-result layout as above, 4 or 8 waves.  A wave owns tiles of 32 keys of the block's
// share (tile i -> wave i % waves).  S^T = K Q^T with v_mfma_f32_16x16x32_bf16, keys as rows: the K
// operand is read from LDS in operand layout (lane l: key l%16, dims 8(l/16)..+7 of a 32-dim chunk).  A lane then holds 4+4 keys of ONE head (l%16), so the running softmax needs two
// cross-lane steps.  O^T = V^T P^T: P^T is already the B operand (slot (l/16, e) stands for key
// 4(l/16) + e of the first 16 keys for e < 4, of the second 16 for e >= 4); V goes through LDS too
// (written as rows, read as columns with ds_read_b64_tr_b16).  16x16x32 layout: A[i = l%16][k = 8(l/16)..+7],
// B[k = 8(l/16)..+7][j = l%16], D[i = 4(l/16) + e][j = l%16].
//
// What bounds a block is the chain of one tile's steps in a wave, not memory (two tiles in flight gain nothing): scalar loop
// control, accumulators in plain vector registers (two waves a SIMD asked for), one multiplication for a key's page, lane groups
// that meet by register swaps, a sum that meets only at the end and no rescaling where no maximum grew took a tile from 1.25 to
// 0.85 us.  24:8 heads of 64: 40 rows of 100..2,048 keys 25.1 -> 20.2 us, one row of 258 keys 6.7 -> 5.7; 32:2 heads of 128: 4 rows
// of 16,385 keys 24.0 -> 21.2, 60 rows of 100..8,000 keys 49.9 -> 43.
typedef __bf16 gq_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gq_v4f __attribute__((ext_vector_type(4)));
typedef float gq_v8f __attribute__((ext_vector_type(8)));
typedef short gq_v4s __attribute__((ext_vector_type(4)));
constexpr int kGqaKeys = 32;

union GqFrag {
    uint4 u;
    uint16_t h[8];
    gq_bf16x8 v;
};

template <int DH, bool STAGED, int WV>
__global__ void __launch_bounds__(64 * WV, 2)
attn_decode_gqa_kernel(const uint16_t* __restrict__ q, int q_stride,
                       const uint16_t* __restrict__ kcache, const uint16_t* __restrict__ vcache,
                       const int* __restrict__ block_tables, int bt_stride,
                       const int* __restrict__ tok_list, const int* __restrict__ token_req,
                       const int* __restrict__ positions,
                       float* __restrict__ part_acc, float* __restrict__ part_ml,
                       int nh, int nkvh, int page_size, float scale, int window, int nsplit, unsigned page_rcp,
                       uint16_t* __restrict__ final_out, int out_stride) {
    constexpr int NC = DH / 32;                    // 32-dim chunks of the score product
    constexpr int ND = DH / 16;                    // 16-dim chunks of the output
    constexpr int VS = DH + 8;                     // LDS row stride of a V tile (elements)
    constexpr int NV = kGqaKeys * (DH / 8) / 64;   // 16-byte V loads per lane and tile
    __shared__ __attribute__((aligned(16))) uint16_t Vs[WV][kGqaKeys * VS];
    __shared__ float sm_ml[WV][16][2];
    __shared__ int pages[kDecMaxPages];
    static_assert(sizeof(uint16_t) * kGqaKeys * VS >= sizeof(float) * 16 * DH, "merge buffer fits in the V tiles");
    float* sm_o = reinterpret_cast<float*>(&Vs[0][0]);       // [waves][16 heads][DH] after the key loop

    const int split = blockIdx.x, kvh = blockIdx.y, n = blockIdx.z;
    const int t = tok_list ? tok_list[n] : n;
    const int g = nh / nkvh;
    const int pos = positions[t];
    const int* bt = block_tables + (size_t)token_req[t] * bt_stride;
    const int lo0 = (window > 0 && pos - window + 1 > 0) ? pos - window + 1 : 0;
    const int nkeys = pos + 1 - lo0;
    const int per = (nkeys + nsplit - 1) / nsplit;
    const int lo = lo0 + split * per;
    int hi = lo + per;
    if (hi > pos + 1) hi = pos + 1;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float scale2 = scale * 1.4426950408889634f;   // scores and running maxima in units of log 2: exp2 is one instruction
    const int lr = lane & 15, lg = lane >> 4;      // row / column of a tile, and the lane group
    const size_t head_stride = (size_t)page_size * DH;
    const size_t page_stride = (size_t)nkvh * head_stride;
    const uint16_t* kbase = kcache + (size_t)kvh * head_stride;
    const uint16_t* vbase = vcache + (size_t)kvh * head_stride;

    auto page_of = [&](int key) { return STAGED ? (int)__umulhi((unsigned)key, page_rcp) : key / page_size; };
    const int page_lo = page_of(lo);
    const int n_pages = (hi > lo) ? page_of(hi - 1) - page_lo + 1 : 0;
    if (STAGED)
        for (int i = threadIdx.x; i < n_pages; i += 64 * WV) pages[i] = bt[page_lo + i];
    __syncthreads();
    auto row_of = [&](int key) -> size_t {
        const int lp = page_of(key);
        const int pg = STAGED ? pages[lp - page_lo] : bt[lp];
        return (size_t)pg * page_stride + (size_t)(key - lp * page_size) * DH;
    };

    const int n_tiles = (hi > lo) ? (hi - lo + kGqaKeys - 1) / kGqaKeys : 0;

    for (int h0 = 0; h0 < g; h0 += 16) {
        // Q^T operand: head lr of this chunk, dims 32c + 8 lg .. +7
        GqFrag qf[NC];
        {
            const bool head_ok = h0 + lr < g;
            const uint16_t* qp = q + (size_t)t * q_stride + (size_t)(kvh * g + h0 + (head_ok ? lr : 0)) * DH + 8 * lg;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                if (head_ok) qf[c].u = *reinterpret_cast<const uint4*>(qp + 32 * c);
                else qf[c].u = make_uint4(0, 0, 0, 0);
            }
        }
        gq_v4f oacc[ND];
#pragma unroll
        for (int c = 0; c < ND; ++c) oacc[c] = gq_v4f{0.f, 0.f, 0.f, 0.f};
        float m = -INFINITY, l = 0.f;              // of head lr, the same in the four lane groups

        // Keys and values are read in whole rows (consecutive lanes take consecutive 16-byte pieces, so a wave's load
        // covers whole cache lines) with loads the caches do not keep.  The keys then pass through the wave's LDS tile
        // into operand layout (key 16 s2 + lr, dims 32 c + 8 lg .. +7) before the values take the tile over: loaded
        // straight in operand layout a wave's load covered 64 bytes of each of 16 rows, half a line.
        uint4 kraw[NV], vreg[NV];
        constexpr int KPI = 512 / DH;              // keys a wave's load covers
        const int key0 = lane / (DH / 8), oct = lane % (DH / 8);
        // No condition around a load: keys beyond the share read its last key.
        auto fetch = [&](int tile) {
            const int kt = lo + tile * kGqaKeys + key0;
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const size_t at = row_of(min(kt + KPI * i, hi - 1)) + oct * 8;
                kraw[i] = load_stream16(kbase + at);
                vreg[i] = load_stream16(vbase + at);
            }
        };
        uint16_t* const mine = &Vs[wave][key0 * VS + oct * 8];
        auto stash = [&](const uint4* regs) {
#pragma unroll
            for (int i = 0; i < NV; ++i) *reinterpret_cast<uint4*>(mine + KPI * i * VS) = regs[i];
        };
        // A wave writes and reads only its own tile in LDS, and LDS serves a wave's instructions in order, so no
        // block barrier is needed in this loop (wave_barrier keeps the compiler from moving LDS accesses across it).
        if (wave < n_tiles) fetch(wave);
        for (int tile = wave; tile < n_tiles; tile += WV) {
            const int kt = lo + tile * kGqaKeys;
            const bool last = kt + kGqaKeys > hi;
            GqFrag kreg[2][NC];
            __builtin_amdgcn_wave_barrier();
            stash(kraw);
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    kreg[s2][c].u = *reinterpret_cast<const uint4*>(&Vs[wave][(16 * s2 + lr) * VS + 32 * c + 8 * lg]);
            if (last) {                             // stand-ins for keys beyond the share: weight 0, but 0 * infinity is NaN
#pragma unroll
                for (int i = 0; i < NV; ++i)
                    if (kt + key0 + KPI * i >= hi) vreg[i] = make_uint4(0, 0, 0, 0);
            }
            __builtin_amdgcn_wave_barrier();
            stash(vreg);
            __builtin_amdgcn_wave_barrier();
            if (tile + WV < n_tiles) fetch(tile + WV);      // the next tile's loads fly during the rest of this one

            // ---- S^T = K Q^T, two subtiles of 16 keys ----------------------------------
            gq_v4f sacc[2];
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                sacc[s2] = gq_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    sacc[s2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kreg[s2][c].v, qf[c].v, sacc[s2], 0, 0, 0);
            }
            float sv[8], mloc = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; ++e) sv[e] = sacc[e >> 2][e & 3] * scale2;       // in units of log 2
            if (last) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (kt + 16 * (e >> 2) + 4 * lg + (e & 3) >= hi) sv[e] = -INFINITY;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) mloc = fmaxf(mloc, sv[e]);
            mloc = swap_max<16>(swap_max<32>(mloc));
            if (__builtin_amdgcn_ballot_w64(mloc > m)) {     // rescaled only where a maximum grew; a row's largest weight stays exactly 1
                const float m_new = fmaxf(m, mloc);
                const float corr = __builtin_amdgcn_exp2f(m - m_new);
                l *= corr;
                m = m_new;
#pragma unroll
                for (int c = 0; c < ND; ++c) oacc[c] *= corr;
            }
            gq_v8f pf;
            float rs = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) { const float p = __builtin_amdgcn_exp2f(sv[e] - m); pf[e] = p; rs += p; }
            l += rs;                                // of this lane's keys; the lane groups meet after the loop
            const gq_bf16x8 pb = __builtin_convertvector(pf, gq_bf16x8);

            // ---- O^T += V^T P^T ----------------------------------------------------------------
            // V^T operand by transposing LDS reads: lane 16 G + i receives, for e = 0..3, element i % 4 of the
            // 8-byte chunk that lane 16 G + i / 4 + 4 e pointed at; this lane points at key 4 lg + lr / 4 (and 16
            // keys on), dims 16 c + 4 (lr % 4) ..+3, and gets dim 16 c + lr of keys 4 lg + e (and 16 keys on)
            const uint16_t* vrow = &Vs[wave][(4 * lg + (lr >> 2)) * VS + 4 * (lr & 3)];
#pragma unroll
            for (int c = 0; c < ND; ++c) {
                const gq_v4s lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gq_v4s __attribute__((address_space(3)))*)(vrow + 16 * c));
                const gq_v4s hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gq_v4s __attribute__((address_space(3)))*)(vrow + 16 * VS + 16 * c));
                const auto both = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
                oacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gq_bf16x8, both), pb, oacc[c], 0, 0, 0);
            }
        }
        l = swap_add<16>(swap_add<32>(l));

        // ---- merge the four waves; O^T[d = 16c + 4 lg + e][head lr] ---------------------------
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ND; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) sm_o[(wave * 16 + lr) * DH + 16 * c + 4 * lg + e] = oacc[c][e];
        if (lg == 0) { sm_ml[wave][lr][0] = m; sm_ml[wave][lr][1] = l; }
        __syncthreads();
        for (int idx = threadIdx.x; idx < 16 * DH; idx += 64 * WV) {
            const int j = idx / DH, d = idx - j * DH;
            if (h0 + j >= g) continue;
            float mm = -INFINITY;
            for (int w = 0; w < WV; ++w) mm = fmaxf(mm, sm_ml[w][j][0]);
            float a = 0.f, ll = 0.f;
            if (mm != -INFINITY) {
                for (int w = 0; w < WV; ++w) {
                    const float cw = __builtin_amdgcn_exp2f(sm_ml[w][j][0] - mm);
                    a += sm_o[(w * 16 + j) * DH + d] * cw;
                    ll += sm_ml[w][j][1] * cw;
                }
            }
            const int h = kvh * g + h0 + j;
            if (final_out) {                        // a single split: this is the result, no second pass
                final_out[(size_t)t * out_stride + (size_t)h * DH + d] = f32_to_bf16_bits(a / ll);
                continue;
            }
            const size_t pidx = ((size_t)n * nh + h) * nsplit + split;
            part_acc[pidx * DH + d] = a;
            if (d == 0) { part_ml[pidx * 2] = mm * 0.6931471805599453f; part_ml[pidx * 2 + 1] = ll; }   // natural units for the second pass
        }
        __syncthreads();                            // sm_o (the V tiles) is reused by the next chunk
    }
}

// Grouped queries in bfloat16 run the matrix-core kernel: the one place that says so (the key-split rule asks here too).
IC_EXPORT int ic_attn_decode_on_matrix_cores(int dtype, int n_heads, int n_kv_heads) { return dtype == IC_BF16 && n_heads != n_kv_heads; }

template <typename T, int DH>
static int launch_decode(const void* q, int q_stride, void* out, int out_stride, const void* kcache,
                         const void* vcache, const int* block_tables, int bt_stride, const int* tok_list,
                         const int* token_req, const int* positions, float* part_acc, float* part_ml,
                         int n_tok, int nh, int nkvh, int page_size, float scale, int window, int nsplit,
                         hipStream_t stream) {
    dim3 grid(nsplit, nkvh, n_tok), block(kDecThreads);
    // A block never needs more page ids than a request has.  The multiplication that stands for a division by the page size is exact
    // for keys below 2^32 / page_size, which kDecMaxPages pages of fewer than 2,048 keys stay below.
    const bool staged = bt_stride <= kDecMaxPages && page_size >= 2 && page_size < 2048;
    const unsigned page_rcp = (unsigned)(((1ull << 32) + page_size - 1) / page_size);
    void* direct = (nsplit == 1) ? out : nullptr;       // one split writes the result itself
#define IC_DEC_LAUNCH(KERNEL, TQ)                                                                           \
    hipLaunchKernelGGL(KERNEL, grid, block, 0, stream, (const TQ*)q, q_stride, (const TQ*)kcache,           \
                       (const TQ*)vcache, block_tables, bt_stride, tok_list, token_req, positions, part_acc, \
                       part_ml, nh, nkvh, page_size, scale, window, nsplit, page_rcp, (TQ*)direct, out_stride)
    if (ic_attn_decode_on_matrix_cores(sizeof(T) == 2 ? IC_BF16 : IC_F32, nh, nkvh)) {
        // Eight waves where one split's share is long for four and the blocks are too few to fill the units anyway (24:8 heads of 64,
        // one split: 258 keys 6.1 -> 5.8 us, 16 rows of up to 2,000 keys 18.6 -> 14.1; with 320 pairs of 1,000 keys 19.2 -> 21.1).
        // Heads of 128 and shares of several splits gain nothing by them (32:2 heads, 16,385 keys in 32 splits: 21.6 and 21.3).
        const bool eight = DH == 64 && nsplit == 1 && n_tok * nkvh <= 128;
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

// Whether a step of n_rows single tokens, all its rows, is worth the kernel above (2 us a step): 64 rows of 36 heads of 64 over 300..2,100
// keys 94.8 -> 89.1 us a layer, 40 rows of 24:8 heads over 100..2,048 22.2 -> 20.2, 24 rows of 36 heads over 100..1,500 27.4 -> 25.7.  Several
// splits balance the walks already (16 rows of 36 heads in 4 splits 26.7 and 28.2), and up to one block a unit all start at once.
IC_EXPORT int ic_attn_decode_wants_order(int n_rows, int nkvh, int nsplit, int compute_units) {
    return nsplit == 1 && n_rows > 1 && n_rows <= kOrderRows && (long long)n_rows * nkvh > (compute_units > 0 ? compute_units : 256);
}

IC_EXPORT int ic_attn_decode_order(const int* positions, int* order, int n_rows, hipStream_t stream) {
    if (n_rows <= 0) return IC_OK;
    if (n_rows > kOrderRows || !positions || !order) return IC_ERR_ARG;
    hipLaunchKernelGGL(attn_decode_order_kernel, dim3(1), dim3((n_rows + 63) / 64 * 64), 0, stream, positions, order, n_rows);
    return ic_launch_status();
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
