// The blocks of the kernels of single tokens, for the kernels of attn_decode.hip and the one of attn_mixed.hip that runs them beside blocks of
// prompt tiles.
#pragma once
#include "common.h"

constexpr int kDecThreads = 256;
constexpr int kDecWaves = kDecThreads / 64;
constexpr int kDecUnroll = 4;
constexpr int kDecMaxPages = 1024;   // page ids of one block's keys staged in LDS (else read from memory)

// key / page_size for any page size and any key below 2^31 - 1 by one multiplication and a shift (a division is some 20 instructions).
// With 2^shift <= page_size < 2^(shift + 1) and mul = floor((2^(32 + shift) - 1) / page_size), (key + 1) mul / 2^(32 + shift) lies below
// (key + 1) / page_size by less than 1 / page_size and by more than nothing, so its whole part is key / page_size.  Against the division, 32 float32 rows
// of 24:8 heads over 100..2,000 keys: 36.5 -> 33.5 us with pages of 64, 37.4 -> 34.3 with pages of 2,048.
struct PageDivider {
    unsigned mul;
    int shift;
    explicit PageDivider(int page_size) : shift(31 - __builtin_clz((unsigned)page_size)) { mul = (unsigned)(((1ull << (32 + shift)) - 1) / (unsigned)page_size); }
    __host__ __device__ __forceinline__ int page_of(int key) const {
        return (int)((unsigned)(((unsigned long long)(unsigned)key * mul + mul) >> 32) >> shift);
    }
};

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

// merge running-softmax state b into a (which product of a sum is rounded first is written out: left to the compiler it differs from kernel to kernel)
__device__ __forceinline__ void merge_state(float& m, float& l, float* acc, int n,
                                            float mb, float lb, const float* accb) {
    const float mn = fmaxf(m, mb);
    if (mn == -INFINITY) return;                 // both empty
    const float ca = __builtin_amdgcn_exp2f(m - mn), cb = __builtin_amdgcn_exp2f(mb - mn);   // maxima in units of log 2
    l = fmaf(lb, cb, l * ca);
    for (int i = 0; i < n; ++i) acc[i] = fmaf(acc[i], ca, accb[i] * cb);
    m = mn;
}

template <typename T, int DH, int GQ, bool STAGED>
__device__ __forceinline__ void split_block(const T* __restrict__ q, int q_stride,
                         const T* __restrict__ kcache, const T* __restrict__ vcache,
                         const int* __restrict__ block_tables, int bt_stride,
                         const int* __restrict__ tok_list, const int* __restrict__ token_req,
                         const int* __restrict__ positions,
                         float* __restrict__ part_acc, float* __restrict__ part_ml,
                         int nh, int nkvh, int page_size, float scale, int window, int nsplit, PageDivider div,
                         T* __restrict__ final_out, int out_stride,
                         const int split, const int kvh, const int n, float (*const sm_acc)[GQ][DH], float (*const sm_ml)[GQ][2], int* const pages) {
    constexpr int VEC = Vec16<T>::N;
    constexpr int LPK = DH / VEC;                 // lanes per key
    constexpr int KPW = 64 / LPK;                 // keys per wave per step
    constexpr int KPB = KPW * kDecWaves;          // keys per block per step
    static_assert(DH % VEC == 0 && 64 % LPK == 0, "head size must split a wave evenly");

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
    auto page_of = [&](int key) { return div.page_of(key); };
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
                const float mb = lane_xor(m[j], o);
                const float lb = lane_xor(l[j], o);
                float ab[VEC];
#pragma unroll
                for (int i = 0; i < VEC; ++i) ab[i] = lane_xor(acc[j][i], o);
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
// that meet by register swaps, a sum that meets only at the end and no rescaling where no maximum grew took a tile from 1.16 to
// 0.83 us (heads of 128: 1.93 to 1.13).  24:8 heads of 64: 40 rows of 100..2,048 keys 25.6 -> 22.3 us as they lie (20.4 the longest first), one row of
// 258 keys 6.7 -> 5.7 (with eight waves); 32:2 heads of 128: 4 rows of 16,385 keys 24.1 -> 22.2, 60 rows of 100..8,000 keys 49.7 -> 43.4.
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

// LDS of a block: tiles of V (gqa_tile_elements<DH, WV>() elements), states of the waves, page ids.
template <int DH, int WV> constexpr int gqa_tile_elements() { return WV * kGqaKeys * (DH + 8); }

template <int DH, bool STAGED, int WV>
__device__ __forceinline__ void gqa_block(const uint16_t* __restrict__ q, int q_stride,
                       const uint16_t* __restrict__ kcache, const uint16_t* __restrict__ vcache,
                       const int* __restrict__ block_tables, int bt_stride,
                       const int* __restrict__ tok_list, const int* __restrict__ token_req,
                       const int* __restrict__ positions,
                       float* __restrict__ part_acc, float* __restrict__ part_ml,
                       int nh, int nkvh, int page_size, float scale, int window, int nsplit, PageDivider div,
                       uint16_t* __restrict__ final_out, int out_stride,
                       const int split, const int kvh, const int n, uint16_t* const Vs, float (*const sm_ml)[16][2], int* const pages) {
    constexpr int NC = DH / 32;                    // 32-dim chunks of the score product
    constexpr int ND = DH / 16;                    // 16-dim chunks of the output
    constexpr int VS = DH + 8;                     // LDS row stride of a V tile (elements)
    constexpr int NV = kGqaKeys * (DH / 8) / 64;   // 16-byte V loads per lane and tile
    static_assert(sizeof(uint16_t) * kGqaKeys * VS >= sizeof(float) * 16 * DH, "merge buffer fits in the V tiles");
    float* sm_o = reinterpret_cast<float*>(Vs);          // [waves][16 heads][DH] after the key loop

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

    auto page_of = [&](int key) { return div.page_of(key); };
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
        uint16_t* const mine = Vs + wave * (kGqaKeys * VS) + key0 * VS + oct * 8;
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
                    kreg[s2][c].u = *reinterpret_cast<const uint4*>(Vs + wave * (kGqaKeys * VS) + (16 * s2 + lr) * VS + 32 * c + 8 * lg);
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
            const uint16_t* vrow = Vs + wave * (kGqaKeys * VS) + (4 * lg + (lr >> 2)) * VS + 4 * (lr & 3);
#pragma unroll
            for (int c = 0; c < ND; ++c) {
                const gq_v4s lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gq_v4s __attribute__((address_space(3)))*)(vrow + 16 * c));
                const gq_v4s hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((gq_v4s __attribute__((address_space(3)))*)(vrow + 16 * VS + 16 * c));
                const auto both = __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7);
                oacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gq_bf16x8, both), pb, oacc[c], 0, 0, 0);
            }
        }
        l = swap_add<16>(swap_add<32>(l));

        // ---- merge the waves; O^T[d = 16c + 4 lg + e][head lr] ---------------------------
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
