// Attention of prompt portions over the paged cache in float32 on the bfloat16 matrix cores, every number in three parts (float_parts.h).
//
// A block of four waves owns up to 128 consecutive tokens of one request and one head and walks the keys 64 or 128 at a time through LDS, as the bfloat16
// kernel does; the tile list is the same.  Scores are computed transposed, S^T = K Q^T, so a lane holds 16 keys of ONE query and the running softmax needs a single
// cross-lane step; the probabilities are then already the B operand of O^T = V^T P^T.  Keys and values are split once per block, on their way from registers to LDS
// (rows of bfloat16 a part); queries once, probabilities by the wave that made them.  The softmax and every sum stay float32.
//
// 32x32x16 operand layout (lane l, h = l / 32): A[i = l % 32][k = 8 h .. 8 h + 7], B[k][j = l % 32], D[i = 8 (r / 4) + 4 h + r % 4][j = l % 32] for the 16
// accumulators r.  In O^T = V^T P^T slot (h, e) of a chunk of 16 keys stands for key 4 h + e (e < 4) or 8 + 4 h + e - 4, where D left P^T; V^T is read with
// ds_read_b64_tr_b16, which transposes on the way out of LDS (attn_prefill_mfma.h).
//
// Six bfloat16 products take 0.375 of the time of v_mfma_f32_32x32x2_f32, the float32 instruction, and with that a step's products no longer bound the kernel: a step of
// 32 keys a wave takes 3.2 us where it is alone on its SIMD, 0.65 of it products.  With float32 instructions / so, us (one block's keys by themselves in
// registers, lookups in a chain, the way before): 24:8 heads of 64, 509 tokens after 130 33 / 26; 100 after 900 45 / 31; 4,000 548 / 298; 12 portions of
// 40 after 700 99 / 44; 36:36, 300 after 130 30 / 25; 32:2 of 128, 300 after 130 47 / 39; 2,048 424 / 238; 4,000 1,282 / 886, in a window of 300 269 / 229.  Heads of 128 have one
// block a unit, where 32-bit operands left room for two: 40 portions of two tokens of 32 heads 43 / 41.  Error against 64 bits (relative, 2-norm)
// 1.4..2.9e-7, with float32 instructions 2.0..4.3e-7.
//
// A block that ends with a result that is not finite, or under 2^-64 (PartsCheck), walks again with the float32
// instructions, whose two values of the summed dimension per instruction are free as long as A and B agree: in S^T = K Q^T instruction c takes head
// dims c and c + DH / 2, in O^T = V^T P^T accumulator r of S^T is the B operand as it stands.
//
// Every SIMD needs some work: with few tiles (a portion of 512 tokens of 24 heads makes 96) a block takes only 64 or 32 of a tile's rows and its waves
// share the keys between them, KG key groups of 32 keys a step, merged through LDS at the end.  The next step's keys and values are on their way in registers
// while this one's are used.
//
// Cache layout of one layer: K and V planes [num_pages, n_kv_heads, page_size, head_dim].
#include "common.h"
#include "float_parts.h"

typedef parts_v4f f32_v4;
typedef short f32_tr4 __attribute__((ext_vector_type(4)));
typedef float f32_v16 __attribute__((ext_vector_type(16)));

constexpr int kF32Threads = 256;
constexpr int kF32Rows = 128;     // query rows per block (must equal the bfloat16 kernel's tile height: one tile list serves both)

// KG key groups: 1 (a step of 64 keys, every wave all of them), 2 (64 keys, 32 a group) or 4 (128 keys, 32 a group).
template <int DH, int KG>
__global__ void __launch_bounds__(kF32Threads, DH == 128 ? 1 : 2)
attn_prefill_f32_kernel(const float* __restrict__ q, int q_stride, float* __restrict__ out, int out_stride,
                        const float* __restrict__ kcache, const float* __restrict__ vcache,
                        const int* __restrict__ block_tables, int bt_stride, const int4* __restrict__ tiles,
                        int n_tiles, int nh, int nkvh, int page_shift, float scale_log2e, int window) {
    constexpr int HALF = DH / 2;          // float32 matrix instructions per 32-key tile of S^T
    constexpr int ND = DH / 32;           // 32-row tiles of O^T
    constexpr int KS = DH + 4;            // row stride of the K tile (floats): 16-byte reads of 16 consecutive rows cover all banks
    constexpr int VS = DH + 8;            // row stride of the V tile: rows four apart (the wave's two halves) fall into different banks
    constexpr int KEYS = KG == 4 ? 128 : 64;                  // keys per step
    constexpr int GK = KG == 1 ? 64 : 32;                     // of them, a group's
    constexpr int NT = GK / 32;                               // 32-key tiles of a group
    constexpr int RW = 4 / KG;                                // waves that own rows, 32 each
    constexpr int NL = KEYS * (DH / 8) / kF32Threads;         // pairs of 16-byte loads per thread and plane
    constexpr int MF = 2 + ND * 16;                           // floats a lane hands over at the end
    constexpr int PKS = DH + 8, PVS = DH + 16;                // row strides of the parts' K and V tiles (bfloat16), for 16-byte reads of 16 rows and 8-byte reads of 4 x 32 bytes
    // With four groups the values' parts take the keys' place when those have been read, so that two blocks fit a unit: 24:8 heads of 64, 509 tokens after 130
    // 30.3 -> 23.2 us, alone on its unit (100 after 900) 29.1 -> 29.6.
    constexpr bool SHARED = KG == 4;
    constexpr int PART_FLOATS = 3 * KEYS * (SHARED ? PVS : PKS + PVS) / 2, F32_FLOATS = KEYS * (KS + VS);
    constexpr int FLOATS = PART_FLOATS > F32_FLOATS ? PART_FLOATS : F32_FLOATS;
    static_assert(KG == 1 || FLOATS >= (4 - RW) * 64 * MF, "the merge buffer fits in the tiles");
    __shared__ __attribute__((aligned(16))) float tile_mem[FLOATS];
    __shared__ int odd;
    float* const Ks = tile_mem;
    float* const Vs = tile_mem + KEYS * KS;
    uint16_t* const Kp = reinterpret_cast<uint16_t*>(tile_mem);
    uint16_t* const Vp = SHARED ? Kp : Kp + 3 * KEYS * PKS;

    // Tile-major, all heads of the longest tile first.  Heads are innermost: blocks go round the XCDs in turn, and where the tiles are low the row groups that
    // have nothing to do must not all be the same XCDs'.  Nor the same shader engines', where a unit holds one block (heads of 128): there the first row groups of as many
    // tiles as fill the chip come before the second ones.  Portions of two tokens, us: 12 after 2,000 of 16 heads 300 -> 164, 40 after 300 of 8 heads 77 -> 57; elsewhere
    // -4 to +5 %.  Heads of 64, two blocks a unit, lose by it (2,048 tokens of 8 heads 58 -> 75).
    constexpr bool ROUNDS = KG > 1 && DH == 128;
    const int h = (int)blockIdx.x % nh, slot = (int)blockIdx.x / nh;
    const int round = ROUNDS ? (256 + nh - 1) / nh : 1, first = slot / (KG * round) * round;      // tiles of a round, and its first one
    const int in_round = n_tiles - first < round ? n_tiles - first : round, at = slot - KG * first;
    const int sub = ROUNDS ? at / in_round : at;
    const int4 tile = tiles[ROUNDS ? first + at - sub * in_round : first];
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

    f32_v16 oacc[ND];
    float m, l;

    const size_t head_stride = (size_t)page_size * DH;
    const float* kbase = kcache + (size_t)kvh * head_stride;
    const float* vbase = vcache + (size_t)kvh * head_stride;
    const size_t page_stride = (size_t)nkvh * head_stride;

    // A step's keys and values.  The page ids are read a step before, and no load stands under a condition: in a chain of lookups and loads, each waiting for
    // the one before, a step took 1.6 us more.  Keys outside the tile's range, which are masked, are replaced by the nearest inside.
    f32_v4 kr[NL][2], vr[NL][2];
    int page[NL];
    const int load_key = tid / (DH / 8), load_at = tid % (DH / 8) * 8;
    constexpr int KPI = kF32Threads / (DH / 8);               // keys a pass of loads covers
    auto key_of = [&](int kb, int i) {
        const int ka = kb + load_key + i * KPI;
        return ka < first_key ? first_key : ka > last_key ? last_key : ka;
    };
    auto look_up = [&](int kb) {
#pragma unroll
        for (int i = 0; i < NL; ++i) page[i] = bt[key_of(kb, i) >> page_shift];
    };
    auto fetch = [&](int kb) {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const size_t off = (size_t)page[i] * page_stride + (size_t)((key_of(kb, i) & page_mask) * DH + load_at);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                kr[i][e] = *reinterpret_cast<const f32_v4*>(kbase + off + 4 * e);
                vr[i][e] = *reinterpret_cast<const f32_v4*>(vbase + off + 4 * e);
            }
        }
    };
    auto split8 = [](const f32_v4 (&x)[2], parts_v4u (&out)[3]) {
        Split4 half_of[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
#pragma unroll
            for (int k = 0; k < 4; ++k) half_of[e].y[k] = x[e][k];
            each<kSplitSteps>([&](auto o) { split_step<decltype(o)::value>(half_of[e]); });
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) out[p] = parts_v4u{half_of[0].p[p][0], half_of[0].p[p][1], half_of[1].p[p][0], half_of[1].p[p][1]};
    };

    auto walk = [&](auto exact) {
        constexpr bool EXACT = decltype(exact)::value;
        // Q operands, scores in units of log 2 (the softmax scale folded in): Q[query lq][HALF * half + c], or in parts dims 16 c + 8 half .. + 7
        float qf[EXACT ? HALF : 1];
        parts_v4u qp[EXACT ? 1 : DH / 16][3];
        const float* const qrow = q + (size_t)(row0 + (row_ok ? my_row : 0)) * q_stride + (size_t)h * DH;
        if constexpr (EXACT) {
#pragma unroll
            for (int c = 0; c < HALF; c += 4) {
                const f32_v4 v = *reinterpret_cast<const f32_v4*>(qrow + HALF * half + c);
#pragma unroll
                for (int e = 0; e < 4; ++e) qf[c + e] = row_ok ? v[e] * scale_log2e : 0.f;
            }
        } else {
#pragma unroll
            for (int c = 0; c < DH / 16; ++c) {
                f32_v4 x[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    x[e] = *reinterpret_cast<const f32_v4*>(qrow + 16 * c + 8 * half + 4 * e) * scale_log2e;
                    if (!row_ok) x[e] = f32_v4{0.f, 0.f, 0.f, 0.f};
                }
                split8(x, qp[c]);
            }
        }
#pragma unroll
        for (int i = 0; i < ND; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
        m = -INFINITY;
        l = 0.f;
        look_up(kb_begin);
        fetch(kb_begin);
        look_up(kb_begin + KEYS);
        for (int kb = kb_begin; kb <= last_key; kb += KEYS) {
            __syncthreads();                                // the previous step's readers are done
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const int key = load_key + i * KPI;
                if constexpr (EXACT) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        *reinterpret_cast<f32_v4*>(&Ks[key * KS + load_at + 4 * e]) = kr[i][e];
                        *reinterpret_cast<f32_v4*>(&Vs[key * VS + load_at + 4 * e]) = vr[i][e];
                    }
                } else {
                    parts_v4u x[3];
                    split8(kr[i], x);
#pragma unroll
                    for (int p = 0; p < 3; ++p) *reinterpret_cast<parts_v4u*>(&Kp[(p * KEYS + key) * PKS + load_at]) = x[p];
                }
            }
            auto stash_values = [&]() {
#pragma unroll
                for (int i = 0; i < NL; ++i) {
                    parts_v4u x[3];
                    split8(vr[i], x);
#pragma unroll
                    for (int p = 0; p < 3; ++p) *reinterpret_cast<parts_v4u*>(&Vp[(p * KEYS + load_key + i * KPI) * PVS + load_at]) = x[p];
                }
            };
            constexpr bool LATER = SHARED && !EXACT;
            if constexpr (!EXACT && !LATER) stash_values();
            __syncthreads();
            auto send = [&]() {                             // the next step's loads, in flight while this one is used
                if (kb + KEYS <= last_key) { fetch(kb + KEYS); look_up(kb + 2 * KEYS); }
            };
            if constexpr (!LATER) send();
            const int kt = kb + GK * grp;                   // this group's keys
            // is there anything this wave may see?
            const bool seen = wave_ok && kt <= wave_last && !(window > 0 && kt + GK - 1 < wave_first - window + 1);
            // Where the second tile of 32 keys is beyond the wave's last row it is left out: 40 portions of two tokens of 32 heads of 128 50 -> 42 us.
            const int nt_seen = NT > 1 && wave_last - kt < 32 ? 1 : NT;
            f32_v16 sacc[NT];
            if (seen) {
                // ---- S^T = K Q^T : tiles of 32 keys ----------------------------------------------------------
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) sacc[tt][r] = 0.f;
                    if (tt >= nt_seen) continue;                // (masked below)
                    if constexpr (EXACT) {
                        const float* kp = &Ks[(GK * grp + 32 * tt + lq) * KS + HALF * half];
#pragma unroll
                        for (int c = 0; c < HALF; c += 4) {
                            const f32_v4 kx = *reinterpret_cast<const f32_v4*>(kp + c);
#pragma unroll
                            for (int e = 0; e < 4; ++e) sacc[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[e], qf[c + e], sacc[tt], 0, 0, 0);
                        }
                    } else {
                        f32_v16 low;                            // the five smaller products' sum
#pragma unroll
                        for (int r = 0; r < 16; ++r) low[r] = 0.f;
#pragma unroll
                        for (int c = 0; c < DH / 16; ++c) {
                            parts_v8b kx[3];
#pragma unroll
                            for (int p = 0; p < 3; ++p)
                                kx[p] = *reinterpret_cast<const parts_v8b*>(&Kp[(p * KEYS + GK * grp + 32 * tt + lq) * PKS + 16 * c + 8 * half]);
#pragma unroll
                            for (int i = 0; i < kPartTerms; ++i) {
                                const parts_v8b qx = __builtin_bit_cast(parts_v8b, qp[c][kPartY[i]]);
                                if (i < kPartTerms - 1) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kx[kPartX[i]], qx, low, 0, 0, 0);
                                else sacc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kx[kPartX[i]], qx, sacc[tt], 0, 0, 0);
                            }
                        }
                        sacc[tt] += low;
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
                mloc = swap_max<32>(mloc);
                const float m_new = fmaxf(m, mloc);
                const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
                if (__builtin_amdgcn_ballot_w64(mloc > m)) {    // rescaled only where a maximum grew
                    const float corr = exp2f(m - m_use);        // 0 on the first step (m = -inf)
                    l *= corr;
#pragma unroll
                    for (int i = 0; i < ND; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r) oacc[i][r] *= corr;
                    m = m_new;
                }
                float rs = 0.f;
#pragma unroll
                for (int tt = 0; tt < NT; ++tt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float p = __builtin_amdgcn_exp2f(sacc[tt][r] - m_use);
                        sacc[tt][r] = p;
                        rs += p;
                    }
                l += swap_add<32>(rs);
            }
            if constexpr (LATER) {
                __syncthreads();                            // the keys have been read
                stash_values();
                __syncthreads();
                send();
            }
            if (!seen) continue;

            // ---- O^T += V^T P^T : the accumulators of S^T are the B operand as they stand -------------------------------
#pragma unroll
            for (int tt = 0; tt < NT; ++tt) {
                if (tt >= nt_seen) continue;
                if constexpr (EXACT) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float* vp = &Vs[(GK * grp + 32 * tt + 8 * (r >> 2) + 4 * half + (r & 3)) * VS + lq];
#pragma unroll
                        for (int dt = 0; dt < ND; ++dt)
                            oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vp[32 * dt], sacc[tt][r], oacc[dt], 0, 0, 0);
                    }
                } else {
                    // chunks of 16 keys: slot (half, e) is key 4 half + e for e < 4 and 8 + 4 half + e - 4 beyond
#pragma unroll
                    for (int kc = 0; kc < 2; ++kc) {
                        f32_v4 x[2];
#pragma unroll
                        for (int e = 0; e < 8; ++e) x[e / 4][e % 4] = sacc[tt][8 * kc + e];
                        parts_v4u px[3];
                        split8(x, px);
                        const int row = GK * grp + 32 * tt + 16 * kc + 4 * half + ((lane & 15) >> 2);
#pragma unroll
                        for (int dt = 0; dt < ND; ++dt) {
                            parts_v8b vx[3];
#pragma unroll
                            for (int p = 0; p < 3; ++p) {
                                const uint16_t* vp = &Vp[(p * KEYS + row) * PVS + 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3)];
                                const f32_tr4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((f32_tr4 __attribute__((address_space(3)))*)vp);
                                const f32_tr4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((f32_tr4 __attribute__((address_space(3)))*)(vp + 8 * PVS));
                                vx[p] = __builtin_bit_cast(parts_v8b, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
                            }
#pragma unroll
                            for (int i = 0; i < kPartTerms; ++i)
                                oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vx[kPartX[i]], __builtin_bit_cast(parts_v8b, px[kPartY[i]]), oacc[dt], 0, 0, 0);
                        }
                    }
                }
            }
        }
    };
    if (tid == 0) odd = 0;
    walk(std::false_type{});
    PartsCheck check;
    check.add(l);
#pragma unroll
    for (int i = 0; i < ND; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) check.add(oacc[i][r]);
    if (check.failed()) odd = 1;
    __syncthreads();
    if (odd) walk(std::true_type{});

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

// Key groups a block has, from the number of (tile, head) pairs: several until one group's blocks keep the units busy by themselves.  One / two / four groups, us,
// heads of 64: 24 pairs (100 tokens after 900) 57 / 40 / 31; 96 (509 after 130) 38 / 28 / 26; 128 (2,048 of 8 heads) 108 / 76 / 58; 144 (509 after 130 of 36 heads) 38 / 29 / 34;
// 288 (1,000 after 500) 88 / 78 / 97; 432 (12 portions of 40 after 700) 64 / 46 / 67; 576 (2,048) 131 / 134 / 172, (the same in a window of 300) 59 / 55 / 81; 768 (4,000) 298 / 317 / 401.
// Of 128: 32 (100 after 900) 110 / 77; 224 (800 after 200) 111 / 96; 256 (1,000 after 500) 162 / 157, (twice 512 after 512) 114 / 123; 384 (12 portions of 40 after 700) 164 / 120,
// (1,500 after 1,500) 430 / 505; 512 (2,048) 238 / 309.  Over 440 forms (8..64 heads, 1..40 portions of 2..4,000 tokens after 0..3,000, all and a window of 300) no other
// lines do better by more than 0.5 % on average.  Against the float32 instructions throughout: 0.71 of the time for heads of 64, 0.79 of 128, and slower only where a
// walk is one step: 2 tokens after nothing 7.7 -> 8.0 us (64) and 9.6 -> 10.3 (128), 40 such portions of 8 heads 9.4 -> 10.9 and 17.6 -> 19.2.
IC_EXPORT int ic_attn_prefill_f32_groups(int dh, long long pairs) {
    if (dh == 128) return pairs <= 400 ? 2 : 1;
    return pairs <= 128 ? 4 : pairs <= 700 ? 2 : 1;
}

// Called by ic_attn_prefill_split for float32 (attn_prefill_mfma.hip): the arguments are checked there.
int ic_attn_prefill_f32_launch(const void* q, int q_stride, void* out, int out_stride, const void* kcache, const void* vcache,
                               const int* block_tables, int bt_stride, const int* tiles, int n_tiles, int nh, int nkvh, int dh,
                               int page_shift, float scale, int window, hipStream_t stream) {
    if (q_stride % 4 || out_stride % 4 || ((uintptr_t)q & 15) || ((uintptr_t)out & 15) || ((uintptr_t)kcache & 15) ||
        ((uintptr_t)vcache & 15) || ((uintptr_t)tiles & 15))
        return IC_ERR_ARG;
    const float sl2 = scale * 1.4426950408889634f;
    const long long pairs = (long long)nh * n_tiles;
    const int kg = ic_attn_prefill_f32_groups(dh, pairs);
    if (pairs * kg > 0x7fffffffLL) return IC_ERR_ARG;
    dim3 grid((unsigned)nh * (unsigned)n_tiles * (unsigned)kg), block(kF32Threads);
#define IC_F32_LAUNCH(DD, GG)                                                                                                   \
    hipLaunchKernelGGL((attn_prefill_f32_kernel<DD, GG>), grid, block, 0, stream, (const float*)q, q_stride, (float*)out, \
                       out_stride, (const float*)kcache, (const float*)vcache, block_tables, bt_stride,                         \
                       (const int4*)tiles, n_tiles, nh, nkvh, page_shift, sl2, window)
    if (dh == 64) { if (kg == 1) IC_F32_LAUNCH(64, 1); else if (kg == 2) IC_F32_LAUNCH(64, 2); else IC_F32_LAUNCH(64, 4); }
    else if (dh == 128) { if (kg == 1) IC_F32_LAUNCH(128, 1); else IC_F32_LAUNCH(128, 2); }
    else return IC_ERR_UNSUPPORTED;
#undef IC_F32_LAUNCH
    return ic_launch_status();
}
