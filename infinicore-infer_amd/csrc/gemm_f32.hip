// C[M, N] = alpha * A[M, K] * W[N, K]^T in float32 for many rows M, on the bfloat16 matrix cores.
//
// A float32 number is the sum of three bfloat16 numbers: the nearest, the one nearest to what is left, and the rest, which has 7 bits at most; every
// subtraction is exact.  Of the nine products of parts the six of 2^-17 and more are summed in float32, a0 w0 + a0 w1 + a1 w0 + a1 w1 + a0 w2 + a2 w0, the
// small ones first; the three left out are of either sign and 2^-24.2 of a product at most, 2^-27.4 rms, where the rounding of a float32 product is 2^-24 and 2^-25.2.  Six bfloat16 products take 96 cycles where
// the float32 instruction takes 256.  a0 w0 has a sum of its own, which is rounded once per 32 k; the five others are summed beside it.  Error against 64 bits
// (relative, 2-norm; normal values, 1,536 / 3,840 / 5,760 k, 33..2,048 rows): 1.3..2.4e-7 / 1.9..3.9e-7 / 2.3..4.8e-7, the library's float32 product 3.5..7.1e-7 / 0.56..1.1e-6 / 0.67..1.4e-6
// (with all six in one sum 2.9..6.1e-7 / 4.8..9.8e-7).  The 16 rows of a result that is not finite, or under 2^-64, are summed again with
// the float32 instructions (PartsCheck).
//
// A is split once per product, by the norm or the gated unit that computes it or by a kernel before (3.7 us and 10 bytes a value), into the order of the matrix cores' operands: 1 KB per 16 rows, 32 k and part, which go to LDS and
// into registers as they lie.  W stays float32 in memory and in LDS (rows of 128 bytes, the 16-byte chunk c of row r at c ^ (r / 2 % 8)) and is split in registers by the
// one wave that multiplies it: 22 vector instructions per 4 values and 6 MT products, where MT row tiles of 16 share the split.  The matrix cores hide two
// vector instructions per product of 16 cycles (measured: 8.3 ns a product with none to two, 10.3 with three, 12.1 with four), hence no split of A in the loop
// (2.7 per product, 11.5 ns) and blocks of four waves side by side over all rows of the tile, not two by two (W split twice).
// Loads are sent STAGES - 1 stages of 32 k ahead (two stages of 57 KB: 1.7 us a stage that multiplies for 0.85; three of 41 KB: 0.96).
//
// What bounds it: the products' rate, 8.9 ns each (a lone wave a SIMD, power), some 5 us for launch, first loads and way out; the fill of the last round of blocks.  Few rows:
// the weights' bytes.  517 x 7,680 x 1,536: 61.6 us and 4.2 for the split, 1.19 PFLOP/s of parts (library 99); 517 x 1,536 x 3,840 in 4 slices 33.9 (library 61); 2,048 x 7,680 x 1,536 233 (391).
//
// Few tiles: K in slices, blocks of their own, whose sums a second kernel adds up, or the norm that reads them.
#include "common.h"
#include "float_parts.h"
#include "infinicore_infer_variants.h"
#include "workspace_lock.h"

namespace {

typedef parts_v4f v4f;
typedef parts_v4u v4u;
typedef parts_v8b v8b;

struct F32Args {
    const float* A;
    const float* W;
    float* C;                       // slice s at C + s * slice_stride
    const unsigned char* parts;     // A in three parts (split_rows_kernel)
    int M, N, K, lda, ldw, ldc;
    int tiles_m, tiles_n, slices;
    long long slice_stride;
    float alpha;
};

// 16 bytes a lane from base + off to LDS at lds + 16 * lane.
__device__ __forceinline__ void load_to_lds(unsigned lds, unsigned off, const char* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
// waits until at most N of this wave's loads are on their way and all its LDS reads are done
template <int N> __device__ __forceinline__ void wait_loads() {
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (0 << 8));
}

// Ties the accumulators to a place between the products written as assembly, whose results the compiler does not know to wait for.
template <int N, int M> __device__ __forceinline__ void settled(v4f (&acc)[N][M]) {
    asm volatile("s_nop 15");
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int m = 0; m < M; ++m) asm volatile("" : "+a"(acc[n][m]));
    asm volatile("s_nop 7");
}

template <int MT_, int NT_, int STAGES_> struct Shape {
    static constexpr int MT = MT_, NT = NT_, STAGES = STAGES_, BM = 16 * MT, BN = 64 * NT;
    static constexpr int PIECES = 3 * MT + 8 * NT, LOADS = (PIECES + 3) / 4, STAGE_BYTES = 1024 * PIECES;
    static_assert(STAGES >= 2 && STAGES * STAGE_BYTES <= 160 * 1024 && LOADS * (STAGES - 1) < 64, "limits");
};

// What is summed again is bound by the loads' latency.  One row of 517 (130) with a NaN, 7,680 x 1,536: the product 83 -> 114 us (29 -> 57); with a result summed by its lane, k after k,
// 1,623 (526).
// 16 rows of A times NT tiles of 16 rows of W over k0 .. k1 - 1 (multiples of 32) with the float32 instructions: a lane's pointers are at k 4 (lane / 16) of row lane % 16, and
// instruction e takes k e, 4 + e, 8 + e and 12 + e of a run of 16.
template <int NT> __device__ __forceinline__ void sum_again(const float* pa, const float* const (&pw)[NT], int k0, int k1, v4f (&x)[NT]) {
    constexpr int RUNS = NT > 2 ? 4 : 8;
    for (int k = k0; k < k1; k += 16 * RUNS) {
        v4f va[RUNS], vw[NT][RUNS];
#pragma unroll
        for (int u = 0; u < RUNS; ++u) {
            const int from = min(k + 16 * u, k1 - 16);
            va[u] = *reinterpret_cast<const v4f*>(pa + from);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) vw[nt][u] = *reinterpret_cast<const v4f*>(pw[nt] + from);
        }
#pragma unroll
        for (int u = 0; u < RUNS; ++u) {
            if (k + 16 * u >= k1) break;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) x[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vw[nt][u][e], va[u][e], x[nt], 0, 0, 0);
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(256, 1) gemm_f32_kernel(F32Args a) {
    constexpr int MT = T::MT, NT = T::NT, STAGES = T::STAGES, LOADS = T::LOADS, PIECES = T::PIECES;
    __shared__ __attribute__((aligned(1024))) unsigned char lds[STAGES * T::STAGE_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;

    const int tiles = a.tiles_m * a.tiles_n, total = tiles * a.slices;
    const int xcd = blockIdx.x & 7, nth = blockIdx.x >> 3;
    const int v = xcd * (total >> 3) + min(xcd, total & 7) + nth;
    const int slice = v / tiles, t = v - slice * tiles;
    const int bn = t / a.tiles_m, bm = t - bn * a.tiles_m;
    const int m0 = bm * T::BM, n0 = bn * T::BN;
    const int KG = a.K / 32, RT = (a.M + 15) / 16;
    const int s_first = (int)((long long)slice * KG / a.slices), s_end = (int)((long long)(slice + 1) * KG / a.slices), n_stages = s_end - s_first;

    const char* const base_a = (const char*)a.parts + ((size_t)bm * MT * KG + s_first) * 3072;
    const char* const base_w = (const char*)(a.W + (size_t)n0 * a.ldw) + (size_t)s_first * 128;
    // this wave's pieces of a stage: of 1 KB, the rows of A's parts first
    unsigned off[LOADS];
    each<LOADS>([&](auto at) {
        constexpr int I = decltype(at)::value;
        const int piece = min(wave + 4 * I, PIECES - 1);
        if (piece < 3 * MT) {
            const int rt = piece / 3;
            off[I] = (unsigned)min(rt, RT - 1 - bm * MT) * (unsigned)(KG * 3072) + (piece - 3 * rt) * 1024 + lane * 16;
        } else {
            const int row = 8 * (piece - 3 * MT) + (lane >> 3);
            off[I] = (unsigned)min(row, a.N - 1 - n0) * (unsigned)(a.ldw * 4) + 16 * ((lane & 7) ^ ((row >> 1) & 7));
        }
    });
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
    auto fetch = [&](auto at, unsigned s, unsigned into) {
        constexpr int I = decltype(at)::value;
        const int piece = min(wave + 4 * I, PIECES - 1);
        const bool is_a = 4 * I + 3 < 3 * MT || (4 * I < 3 * MT && piece < 3 * MT);
        load_to_lds(into + 1024 * piece, off[I], is_a ? base_a + (size_t)(s * 3072) : base_w + (size_t)(s * 128));
    };
    auto clamped = [&](int s) { return (unsigned)min(s, n_stages - 1); };

    v4f acc[NT][MT], low[NT][MT];                                  // the sums of a0 w0, and of the five smaller products
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = low[nt][mt] = v4f{0.f, 0.f, 0.f, 0.f};

    settled(acc);
    settled(low);
    each<STAGES>([&](auto sc) { each<LOADS>([&](auto i) { fetch(i, clamped(sc), lds0 + decltype(sc)::value * T::STAGE_BYTES); }); });
    const unsigned char* const pa_ = lds + lane * 16;
    const unsigned char* const pw_ = lds + MT * 3072 + (wave * (16 * NT) + r) * 128;
    const int sw = (r >> 1) & 7, place0 = 16 * (kq ^ sw), place1 = 16 * ((4 + kq) ^ sw);
    constexpr int U = 2 * NT;                                      // halves of a wave's operands of W
    v8b pa[2][MT][3];
    Split4 pw[2][U];
    auto w_of = [&](auto uc, auto cur, int buf) {
        constexpr int u = decltype(uc)::value;
        const v4f x = *reinterpret_cast<const v4f*>(pw_ + (u / 2) * 2048 + buf * T::STAGE_BYTES + (u % 2 ? place1 : place0));
#pragma unroll
        for (int e = 0; e < 4; ++e) pw[decltype(cur)::value][u].y[e] = x[e];
    };
    auto a_of = [&](auto ic, auto cur, int buf) {
        constexpr int i = decltype(ic)::value;
        pa[decltype(cur)::value][i / 3][i % 3] = *reinterpret_cast<const v8b*>(pa_ + i * 1024 + buf * T::STAGE_BYTES);
    };
    using Zero = std::integral_constant<int, 0>;
    wait_loads<LOADS * (STAGES - 1)>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    each<3 * MT>([&](auto i) { a_of(i, Zero{}, 0); });
    each<U>([&](auto u) {
        w_of(u, Zero{}, 0);
        each<kSplitSteps>([&](auto o) { split_step<decltype(o)::value, true>(pw[0][decltype(u)::value]); });
    });

    // One k-step of 32: the operands CUR are multiplied; those of the next step are read from LDS and W's split; the loads of stage s + STAGES go out.
    auto step = [&](int s, int buf, auto cur) {
        constexpr int CUR = decltype(cur)::value, P = 6 * MT * NT, D = U < 2 ? U : 2;
        using Next = std::integral_constant<int, CUR ^ 1>;
        const int next = buf + 1 == STAGES ? 0 : buf + 1;
        wait_loads<LOADS * (STAGES - 2)>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const unsigned from = clamped(s + STAGES), into = lds0 + buf * T::STAGE_BYTES;
        each<D>([&](auto u) { w_of(u, Next{}, next); });
        __builtin_amdgcn_sched_barrier(0);
        each<P>([&](auto pc) {
            constexpr int p = decltype(pc)::value, n = p / (6 * MT), term = p / MT % 6, mt = p % MT;
            constexpr auto &X = kPartX, &Y = kPartY;
            const Split4 &lo = pw[CUR][2 * n], &hi = pw[CUR][2 * n + 1];
            const v8b w = __builtin_bit_cast(v8b, v4u{lo.p[X[term]][0], lo.p[X[term]][1], hi.p[X[term]][0], hi.p[X[term]][1]});
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(term == 5 ? acc[n][mt] : low[n][mt]) : "v"(w), "v"(pa[CUR][mt][Y[term]]));
            // the splits are dealt over the products but for the first few, which the reads from LDS have to arrive
            constexpr int HOLD = P / 8, O0 = p < HOLD ? 0 : (p - HOLD) * U * kSplitSteps / (P - HOLD), O1 = p < HOLD ? 0 : (p + 1 - HOLD) * U * kSplitSteps / (P - HOLD);
            constexpr int A0 = p * 3 * MT / P, A1 = (p + 1) * 3 * MT / P, L0 = p * LOADS / P, L1 = (p + 1) * LOADS / P;
            each<A1 - A0>([&](auto k) { a_of(std::integral_constant<int, A0 + decltype(k)::value>{}, Next{}, next); });
            each<L1 - L0>([&](auto k) { fetch(std::integral_constant<int, L0 + decltype(k)::value>{}, from, into); });
            each<O1 - O0>([&](auto k) {
                constexpr int o = O0 + decltype(k)::value, u = o / kSplitSteps;
                if constexpr (o % kSplitSteps == 0 && u + D < U) w_of(std::integral_constant<int, u + D>{}, Next{}, next);
                split_step<o % kSplitSteps, true>(pw[CUR ^ 1][u]);
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        return next;
    };
    int s = 0, buf = 0;
    for (; s + 1 < n_stages; s += 2) {
        buf = step(s, buf, Zero{});
        buf = step(s + 1, buf, std::integral_constant<int, 1>{});
    }
    if (s < n_stages) step(s, buf, Zero{});
    settled(acc);
    settled(low);
    wait_loads<0>();                                               // (nothing may land in LDS after the block)

    float* const C = a.C + (size_t)slice * a.slice_stride;
    const int n_lane = n0 + wave * 16 * NT + 4 * kq;
    auto store = [&](v4f x, int m, int n) {
        float* const to = C + (size_t)m * a.ldc + n;
        x *= a.alpha;
        if (n + 4 <= a.N) *reinterpret_cast<v4f*>(to) = x;
        else
            for (int e = 0; n + e < a.N; ++e) to[e] = x[e];
    };
    unsigned again = 0;                                            // row tiles of this wave that are summed again
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int m = m0 + 16 * mt + r;
        PartsCheck odd;
        if (m < a.M) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int n = n_lane + 16 * nt;
                if (n >= a.N) continue;
                const v4f x = acc[nt][mt] + low[nt][mt];
#pragma unroll
                for (int e = 0; e < 4; ++e) odd.add(x[e]);
                store(x, m, n);
            }
        }
        if (__builtin_amdgcn_ballot_w64(odd.failed())) again |= 1u << mt;
    }
    for (; again; again &= again - 1) {
        const int m = m0 + 16 * __builtin_ctz(again) + r;
        v4f x[NT];
        const float *pa1 = a.A + (size_t)min(m, a.M - 1) * a.lda + 4 * kq, *pw1[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            pw1[nt] = a.W + (size_t)min(n0 + (wave * NT + nt) * 16 + r, a.N - 1) * a.ldw + 4 * kq;
            x[nt] = v4f{0.f, 0.f, 0.f, 0.f};
        }
        sum_again<NT>(pa1, pw1, 32 * s_first, 32 * s_end, x);
        if (m >= a.M) continue;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
            if (n_lane + 16 * nt < a.N) store(x[nt], m, n_lane + 16 * nt);
    }
}

// The rows of A in three parts, in the order of the matrix cores' operands: [row / 16][k / 32][part][lane][8], lane l row l % 16, k 4 (l / 16) .. + 3 and 16 on.
__global__ void __launch_bounds__(256) split_rows_kernel(const float* A, int lda, int M, int K, uint4* out) {
    const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4, KG = K / 32;
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6), rt = w / KG, kg = w - rt * KG;
    if (rt >= (M + 15) / 16) return;
    const float* const from = A + (size_t)min(16 * rt + r, M - 1) * lda + 32 * kg + 4 * kq;
    Split4 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const v4f x = *reinterpret_cast<const v4f*>(from + 16 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[h].y[e] = x[e];
        each<kSplitSteps>([&](auto o) { split_step<decltype(o)::value>(s[h]); });
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) out[(size_t)w * 192 + p * 64 + lane] = uint4{s[0].p[p][0], s[0].p[p][1], s[1].p[p][0], s[1].p[p][1]};
}

// SwiGLU of gate_up [M, 2 di] (gate, then up), as float32 rows and in three parts as above.  One pass where the unit's kernel and the split of its result were two: 517 x 3,840
// 6.6 + 5.5 -> 8.5 us.  (Rows of 16 and 32 k a wave, as the split, so that the parts leave in whole lines.)
__global__ void __launch_bounds__(256) swiglu_parts_kernel(const float* gate_up, float* act, int M, int di, uint4* out) {
    const int lane = threadIdx.x & 63, r = lane & 15, kq = lane >> 4, KG = di / 32;
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6), rt = w / KG, kg = w - rt * KG;
    if (rt >= (M + 15) / 16) return;
    const int row = min(16 * rt + r, M - 1), k = 32 * kg + 4 * kq;
    const float* const from = gate_up + (size_t)row * 2 * di + k;
    Split4 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const v4f g = *reinterpret_cast<const v4f*>(from + 16 * h), u = *reinterpret_cast<const v4f*>(from + di + 16 * h);
        v4f o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = g[e] / (1.0f + expf(-g[e]));
            s[h].y[e] = o[e] = u[e] * x;
        }
        if (16 * rt + r < M) *reinterpret_cast<v4f*>(act + (size_t)row * di + k + 16 * h) = o;
        each<kSplitSteps>([&](auto o) { split_step<decltype(o)::value>(s[h]); });
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) out[(size_t)w * 192 + p * 64 + lane] = uint4{s[0].p[p][0], s[0].p[p][1], s[1].p[p][0], s[1].p[p][1]};
}

// x += alpha * the sum of the slices y [S][M][d]; out = rmsnorm(x) * w, as rows and (parts given) in three parts for the product that follows: one kernel where the sum of the
// slices, the norm and the split were three.  Values, and the order of every sum, are those of the three (norm_row_kernel of elementwise.hip: a row to threads * VPT vectors of 4).
// R rows a block: a row's pieces of the parts are 16 bytes, R neighbours' make R times as many in a line.  Bound by latency: one trip to memory for x and y, the sum across the
// row, the way out.  517 x 1,536, every second one with the down product's slices: 5.4 + 5.5 (and 5.2)
// -> 7.9 us on average; one row a block 8.0.
constexpr int kNormRows = 2;
template <int VPT, int R>
__global__ void __launch_bounds__(1024) norm_parts_kernel(float* x, const float* y, int S, long long stride, float alpha, const float* w, float* out, unsigned char* parts, int M,
                                                          int d, float eps) {
    __shared__ float red[16];
    const int per_row = blockDim.x / R, waves = per_row >> 6, in_block = R == 1 ? 0 : (int)threadIdx.x / per_row;
    const int t = (int)threadIdx.x - in_block * per_row, row = blockIdx.x * R + in_block;
    const bool mine = row < M;
    const size_t at = (size_t)min(row, M - 1) * d;
    v4f v[VPT], wv[VPT];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = 4 * (t + i * per_row);
        v[i] = wv[i] = v4f{0.f, 0.f, 0.f, 0.f};
        if (mine && c < d) {
            wv[i] = *reinterpret_cast<const v4f*>(w + c);
            const v4f xv = *reinterpret_cast<const v4f*>(x + at + c);
            v4f sum = *reinterpret_cast<const v4f*>(y + at + c);
            for (int s = 1; s < S; ++s) sum += *reinterpret_cast<const v4f*>(y + s * stride + at + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] = fmaf(alpha, sum[e], xv[e]);
            *reinterpret_cast<v4f*>(x + at + c) = v[i];
            const float q[4] = {v[i][0], v[i][1], v[i][2], v[i][3]};
            add_squares(ss, q, i == 0);
        }
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float sum = 0.f;
    for (int i = 0; i < waves; ++i) sum += red[in_block * waves + i];
    const float inv = 1.0f / sqrtf(sum / (float)d + eps);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int c = 4 * (t + i * per_row);
        if (c >= d) continue;
        Split4 s;
        v4f o;
#pragma unroll
        for (int e = 0; e < 4; ++e) s.y[e] = o[e] = mine ? v[i][e] * inv * wv[i][e] : 0.f;
        if (mine) *reinterpret_cast<v4f*>(out + at + c) = o;
        if (parts) {                                               // (rows beyond M up to a whole tile of 16: zeros)
            each<kSplitSteps>([&](auto o) { split_step<decltype(o)::value>(s); });
            const int kq = (c >> 2) & 3, h = (c >> 4) & 1;
            unsigned char* const to = parts + ((size_t)(row >> 4) * (d >> 5) + (c >> 5)) * 3072 + ((row & 15) + 16 * kq) * 16 + 8 * h;
#pragma unroll
            for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(to + 1024 * p) = uint2{s.p[p][0], s.p[p][1]};
        }
    }
}

// C = alpha * the sum of the slices P [S][M][N]; N a multiple of 4.
__global__ void __launch_bounds__(256) sum_slices_kernel(const v4f* P, int S, int M, int N4, float* C, int ldc, float alpha) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x, n = (long long)M * N4;
    if (i >= n) return;
    v4f x = P[i];
    for (int s = 1; s < S; ++s) x += P[i + s * n];
    const int m = (int)(i / N4);
    *reinterpret_cast<v4f*>(C + (size_t)m * ldc + 4 * (int)(i - (long long)m * N4)) = alpha * x;
}

template <typename T> int launch(F32Args a, hipStream_t stream) {
    a.tiles_m = (a.M + T::BM - 1) / T::BM;
    a.tiles_n = (a.N + T::BN - 1) / T::BN;
    const long long blocks = (long long)a.tiles_m * a.tiles_n * a.slices;
    if (blocks > (1LL << 30)) return IC_ERR_ARG;
    hipLaunchKernelGGL((gemm_f32_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
    return ic_launch_status();
}

// The shapes of a block, smallest first, and what one costs in microseconds: FIXED + rounds * (ROUND + k-steps of 32 * STAGE * (1 + FULL * x)), x the part of the units
// (256 where this was fitted) that have a block, or the weights' bytes at 6 TB/s where those take longer.  Fitted to 11,700 timed products (13 pairs of N in 512..12,288 and K in
// 768..5,760, 1..2,048 rows, one to four slices, weights out of memory): the shape and slices with the least cost lose 0.5 % to the best on average, 3 % at the 95th percentile.
#define IC_F32_SHAPES(X) \
    /* number, FIXED, STAGE, FULL, ROUND, shape: row tiles of 16, column tiles of 64, stages */ \
    X(0, 1.69, 0.226, 0.13, 1.80, 1, 1, 8) \
    X(1, 1.80, 0.232, 0.26, 2.01, 2, 1, 8) \
    X(2, 1.90, 0.280, 0.15, 2.41, 3, 1, 8) \
    X(3, 1.92, 0.294, 0.20, 2.50, 4, 1, 7) \
    X(4, 1.73, 0.341, 0.20, 2.81, 5, 1, 6) \
    X(5, 1.82, 0.383, 0.22, 3.13, 6, 1, 6) \
    X(6, 1.65, 0.416, 0.26, 3.23, 7, 1, 5) \
    X(7, 1.89, 0.483, 0.23, 3.45, 4, 2, 5) \
    X(8, 1.87, 0.560, 0.24, 3.97, 5, 2, 5) \
    X(9, 1.95, 0.647, 0.24, 4.16, 6, 2, 4) \
    X(10, 1.61, 0.705, 0.28, 4.92, 7, 2, 4) \
    X(11, 1.93, 0.759, 0.29, 5.20, 8, 2, 4) \
    X(12, 1.87, 0.670, 0.23, 4.22, 4, 3, 4) \
    X(13, 1.81, 0.874, 0.24, 5.38, 6, 3, 3) \
    X(14, 1.91, 1.106, 0.28, 6.44, 8, 3, 3)

constexpr int kShapes = 15, kMaxSlices = 4, kFewRows = 32;
struct ShapeCost { int bm, bn; double fixed, stage, full, round; };
constexpr ShapeCost kCosts[kShapes] = {
#define X(I, FIXED, STAGE, FULL, ROUND, MT, NT, ST) {16 * MT, 64 * NT, FIXED, STAGE, FULL, ROUND},
    IC_F32_SHAPES(X)
#undef X
};

double cost_of(const ShapeCost& c, int M, int N, int K, int slices, int units) {
    const double tm = (M + c.bm - 1) / c.bm, x = tm * ((N + c.bn - 1) / c.bn) * slices / units, steps = (double)(K / 32) / slices;
    const double walk = c.fixed + __builtin_ceil(x) * (c.round + steps * c.stage * (1.0 + c.full * (x < 1.0 ? x : 1.0)));
    const double read = 3.0 + 4.0 * N * K * (1.0 + 0.3 * (tm < 5 ? tm - 1 : 4)) / (6e6 * units / 256.0);
    return walk > read ? walk : read;
}

struct Plan { int shape, slices; double cost; };
Plan plan_for(int M, int N, int K, int max_slices, int units) {
    Plan best{-1, 1, 0.0};
    for (int s = 1; s <= max_slices && s <= kMaxSlices && s <= K / 32 && (s == 1 || N % 4 == 0); ++s) {
        const double bytes = 4.0 * M * N, extra = s == 1 ? 0.0 : 3.5 + (s + 1) * bytes / 6e6;
        for (int i = 0; i < kShapes; ++i) {
            const double c = cost_of(kCosts[i], M, N, K, s, units) + extra;
            if (best.shape < 0 || c < best.cost) best = Plan{i, s, c};
        }
    }
    return best;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Whole k-steps, 16-byte pieces of every row, byte offsets within 32 bits.
bool takes(int M, int N, int K, int lda, int ldw, int ldc) {
    if (M <= 0 || M > (1 << 26) || N <= 0 || N > (1 << 30) || K <= 0 || K > (1 << 20) || K % 32 || lda < K || ldw < K || ldc < N || lda % 4 || ldw % 4 || ldc % 4) return false;
    return (long long)ldw * 4 * 192 < (1LL << 32) && (long long)((M + 15) / 16) * (K / 32) < (1LL << 30) && (long long)((M + 15) / 16) * ((N + 63) / 64) * kMaxSlices < (1LL << 30);
}

long long parts_bytes(int M, int K) { return (long long)((M + 15) / 16) * (K / 32) * 3072; }

int split_rows(const float* A, int lda, int M, int K, void* parts, hipStream_t stream) {
    const long long waves = (long long)((M + 15) / 16) * (K / 32);
    hipLaunchKernelGGL(split_rows_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, stream, A, lda, M, K, (uint4*)parts);
    return ic_launch_status();
}

int run(const F32Args& a, int shape, hipStream_t stream) {
    switch (shape) {
#define X(I, FIXED, STAGE, FULL, ROUND, ...) case I: return launch<Shape<__VA_ARGS__>>(a, stream);
        IC_F32_SHAPES(X)
#undef X
    }
    return IC_ERR_ARG;
}

// Rows that are split and multiplied at a time: all, or equal runs of whole row tiles, as many as the workspace holds.
int rows_at_once(int M, int K, long long workspace_bytes) {
    const long long most = workspace_bytes / ((K / 32) * 3072LL) * 16;
    if (most >= M) return M;
    if (most < 16) return 0;
    const long long runs = (M + most - 1) / most;
    return (int)(((M + runs - 1) / runs + 15) / 16 * 16);
}

// ready: A's parts lie in the workspace; keep: slices are left there behind them, not added up.
int product(const float* A, const float* W, float* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int shape, int slices, void* workspace,
            long long workspace_bytes, hipStream_t stream, bool ready = false, bool keep = false) {
    const int at_once = rows_at_once(M, K, workspace_bytes);
    if (at_once <= 0) return IC_ERR_ARG;
    if (slices > 1 && (at_once < M || parts_bytes(M, K) + 4LL * slices * M * N > workspace_bytes)) return IC_ERR_ARG;
    if ((ready || keep) && at_once < M) return IC_ERR_ARG;
    std::lock_guard<std::mutex> lock(workspace_lock());
    for (int m = 0; m < M; m += at_once) {
        const int rows = M - m < at_once ? M - m : at_once;
        const float* const a0 = A + (size_t)m * lda;
        float* const sums = slices > 1 ? (float*)((char*)workspace + parts_bytes(M, K)) : C + (size_t)m * ldc;
        int st = ready ? IC_OK : split_rows(a0, lda, rows, K, workspace, stream);
        if (st) return st;
        st = run(F32Args{a0, W, sums, (const unsigned char*)workspace, rows, N, K, lda, ldw, slices > 1 ? N : ldc, 0, 0, slices, (long long)rows * N,
                         slices > 1 ? 1.0f : alpha}, shape, stream);
        if (st) return st;
    }
    if (slices > 1 && !keep) {
        const long long n = (long long)M * (N / 4);
        if (n > (1LL << 38)) return IC_ERR_ARG;
        hipLaunchKernelGGL(sum_slices_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                           (const v4f*)((const char*)workspace + parts_bytes(M, K)), slices, M, N / 4, C, ldc, alpha);
        return ic_launch_status();
    }
    return IC_OK;
}

int most_slices(int M, int N, int K, long long workspace_bytes) {
    int s = kMaxSlices;                                            // (none where the rows do not fit at once)
    while (s > 1 && parts_bytes(M, K) + 4LL * s * M * N > workspace_bytes) --s;
    return s;
}

// What ic_gemm_f32 costs with this workspace, in microseconds: every run of rows has its split and its product, which reads all of W again.
double cost_with(int M, int N, int K, long long workspace_bytes, int units) {
    const int rows = rows_at_once(M, K, workspace_bytes), runs = (M + rows - 1) / rows;
    return runs * (3.73 + 10.0 * rows * K / (14.8e6 * units / 256.0) + plan_for(rows, N, K, most_slices(M, N, K, workspace_bytes), units).cost);
}

}  // namespace

IC_EXPORT int ic_gemm_f32_supported(int M, int N, int K, int lda, int ldw, int ldc) { return takes(M, N, K, lda, ldw, ldc); }

IC_EXPORT int ic_gemm_f32_takes(int M, int N, int K, int lda, int ldw, int ldc, const void* workspace, long long workspace_bytes) {
    return takes(M, N, K, lda, ldw, ldc) && workspace && aligned16(workspace) && rows_at_once(M, K, workspace_bytes) > 0;
}

IC_EXPORT int ic_gemm_f32_plan_on(int M, int N, int K, int units, int* slices) {
    if (M <= 0 || N <= 0 || K < 32 || units <= 0) return -1;
    const Plan p = plan_for(M, N, K, kMaxSlices, units);
    if (slices) *slices = p.slices;
    return p.shape;
}

// Memory for any plan of the product: A's parts and all slices, up to 64 MB; grows with M.  None where the rule takes the library's product in any case.
IC_EXPORT long long ic_gemm_f32_workspace_bytes(int M, int N, int K) {
    if (M <= kFewRows || N <= 0 || K < 32) return 0;
    const long long need = parts_bytes(M, K) + 4LL * kMaxSlices * M * N, most = 64LL << 20;
    return need < most ? need : most;
}

namespace {

// What the library's float32 product costs, in microseconds: a start, which few k make shorter, and 127 TFLOP/s; no less than 1.4 such starts; and where whole rounds of tiles of
// 64 x 64 cost less, those.  Over 1,134 products (33..2,048 rows, 256..7,680 columns, 256..4,096 k, weights out of memory) and 392 of 32..1,536 k and 32..4,096 columns.
double library_cost(int M, int N, int K, int units) {
    const double start = K < 750 ? 3.3 + 0.0072 * K : 8.7, least = start * 12.0 / 8.7, products = 2.0 * M * N * K / (127e6 * units / 256.0) + start;
    const double rounds = 4.4 + 0.014 * K * __builtin_ceil((double)((M + 63) / 64) * ((N + 63) / 64) / units), whole = products > least ? products : least;
    return rounds < whole ? rounds : whole;
}

}  // namespace

// Whether the split, the product and the sum of its slices beat the library's float32 product; from 33 rows on, since fewer are a matter of the weights' bytes, which it reads as fast
// (8 x 7,680 x 1,536: 13 us, the split alone 4).  Over the 1,134 products above the choice takes 0.907 of the library's time and loses 4 % to the better of the two (the library's choice of
// algorithm is uneven); 28 are 5..35 % slower than the library, most of them of 256..1,024 columns.  130 x 7,680 x 1,536: 33 -> 28, 300 x 2,560 x 1,536: 26 -> 25, 2,048 x 4,096 x 512
// 74 -> 58, on the other side 96 x 2,560 x 1,536: 11 against 16, 1,500 x 512 x 768 13 against 19, 2,048 x 256 x 512 8.5 against 17.  Where the two are near each other parts run,
// whose error is the smaller one.  (Without the rounds, and with 8.7 us as the start for any K, 58 of the 1,134 were over 5 % slower than the library, and 280 products of up to
// 512 k took 1.24 of its time.)  With the workspace there
// is: 64 MB hold 672 rows of 16,384, and 2,048 x 4,096 x 16,384 is four runs of 512 rows (1,403 us, the library 1,798); 16 rows at a time never pay.
IC_EXPORT int ic_gemm_f32_pays_with(int M, int N, int K, long long workspace_bytes, int units) {
    if (M <= kFewRows || N <= 0 || K < 32 || units <= 0 || rows_at_once(M, K, workspace_bytes) <= 0) return 0;
    return cost_with(M, N, K, workspace_bytes, units) < library_cost(M, N, K, units);
}

IC_EXPORT int ic_gemm_f32_pays_on(int M, int N, int K, int units) { return ic_gemm_f32_pays_with(M, N, K, ic_gemm_f32_workspace_bytes(M, N, K), units); }

IC_EXPORT int ic_gemm_f32_pays(int M, int N, int K) { return ic_gemm_f32_pays_on(M, N, K, compute_units()); }

IC_EXPORT long long ic_gemm_f32_parts_bytes(int M, int K) { return M > 0 && K >= 32 ? parts_bytes(M, K) : 0; }

namespace {

bool own_product(const void* A, const void* W, const void* C, int M, int N, int K, int lda, int ldw, int ldc, const void* parts, long long parts_bytes) {
    if (!(M > kFewRows && A && W && C && aligned16(A) && aligned16(W) && aligned16(C) && ic_gemm_f32_takes(M, N, K, lda, ldw, ldc, parts, parts_bytes))) return false;
    const int timed = ic_product_f32_timed(M, N, K, lda, ldw, ldc);
    return (timed >= 0 ? timed : ic_gemm_f32_pays_with(M, N, K, parts_bytes, compute_units())) != 0;
}

}  // namespace

// The product by this file's kernels or the library's, as timed (ic_product_tune) or by the rule: parts is the caller's own memory for the former, workspace the library's.
IC_EXPORT int ic_product_f32(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha, void* parts, long long parts_bytes,
                             void* workspace, long long workspace_bytes, hipStream_t stream) {
    if (own_product(A, W, C, M, N, K, lda, ldw, ldc, parts, parts_bytes)) return ic_gemm_f32(A, W, C, M, N, K, lda, ldw, ldc, alpha, parts, parts_bytes, stream);
    return ic_matmul(A, IC_F32, W, C, IC_F32, M, N, K, lda, ldw, ldc, alpha, workspace, workspace_bytes, stream);
}

// The whole product.  workspace (16-byte aligned): A's parts, or as many rows of them at a time as it holds (16 at least), and the slices where they fit too.
IC_EXPORT int ic_gemm_f32(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha, void* workspace,
                          long long workspace_bytes, hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!A || !W || !C || !workspace || !takes(M, N, K, lda, ldw, ldc) || !aligned16(A) || !aligned16(W) || !aligned16(C) || !aligned16(workspace)) return IC_ERR_ARG;
    const Plan p = plan_for(rows_at_once(M, K, workspace_bytes), N, K, most_slices(M, N, K, workspace_bytes), compute_units());
    return product((const float*)A, (const float*)W, (float*)C, M, N, K, lda, ldw, ldc, alpha, p.shape, p.slices, workspace, workspace_bytes, stream);
}

IC_EXPORT int ic_gemm_f32_cfg(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha, int shape, int slices, void* workspace,
                              long long workspace_bytes, hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!A || !W || !C || !workspace || !takes(M, N, K, lda, ldw, ldc) || !aligned16(A) || !aligned16(W) || !aligned16(C) || !aligned16(workspace) || shape < 0 ||
        shape >= kShapes || slices < 1 || slices > kMaxSlices || slices > K / 32 || (slices > 1 && N % 4)) return IC_ERR_ARG;
    return product((const float*)A, (const float*)W, (float*)C, M, N, K, lda, ldw, ldc, alpha, shape, slices, workspace, workspace_bytes, stream);
}

// Slices of K that ic_product_f32 would use with these arguments where it runs ic_gemm_f32 on all rows at once, else 0.  Then A's parts may be made by what computes A, and the
// slices be added by what reads C.
IC_EXPORT int ic_gemm_f32_whole(const void* A, const void* W, const void* C, int M, int N, int K, int lda, int ldw, int ldc, const void* parts, long long parts_bytes) {
    if (!own_product(A, W, C, M, N, K, lda, ldw, ldc, parts, parts_bytes) || rows_at_once(M, K, parts_bytes) < M) return 0;
    return plan_for(M, N, K, most_slices(M, N, K, parts_bytes), compute_units()).slices;
}

// ic_gemm_f32 of all rows at once.  ready: A's parts lie in the workspace already; keep: more than one slice are left [slice][M][N] at ic_gemm_f32_parts_bytes(M, K) of the
// workspace, and C is not written.
IC_EXPORT int ic_gemm_f32_between(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, void* workspace, long long workspace_bytes, int ready,
                                  int keep, hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!A || !W || !C || !workspace || !takes(M, N, K, lda, ldw, ldc) || !aligned16(A) || !aligned16(W) || !aligned16(C) || !aligned16(workspace)) return IC_ERR_ARG;
    if (rows_at_once(M, K, workspace_bytes) < M) return IC_ERR_ARG;
    const Plan p = plan_for(M, N, K, most_slices(M, N, K, workspace_bytes), compute_units());
    return product((const float*)A, (const float*)W, (float*)C, M, N, K, lda, ldw, ldc, 1.0f, p.shape, p.slices, workspace, workspace_bytes, stream, ready != 0, keep != 0);
}

// Rows of whole k-steps that one block holds.
IC_EXPORT int ic_norm_parts_f32_supported(int d) { return d >= 32 && d % 32 == 0 && d <= 16384; }

// x (float32 [M, d]) += alpha * (the sum of n_slices slices y [M, d], one behind the other); out = rmsnorm(x) * w, in three parts at `parts` too (null: not); all 16-byte aligned.
// y and parts must not overlap.
IC_EXPORT int ic_norm_parts_f32(float* x, const float* y, int n_slices, float alpha, const float* w, float* out, void* parts, int M, int d, float eps, hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!x || !y || !w || !out || n_slices < 1 || n_slices > kMaxSlices || M > (1 << 26) || !ic_norm_parts_f32_supported(d)) return IC_ERR_ARG;
    if (!aligned16(x) || !aligned16(y) || !aligned16(w) || !aligned16(out) || !aligned16(parts)) return IC_ERR_ARG;
    const int vecs = d / 4, t = (vecs + 63) / 64 * 64, per_row = t < 1024 ? t : 1024, vpt = (vecs + per_row - 1) / per_row;
    const int whole = parts ? (M + 15) / 16 * 16 : M, rows = per_row * kNormRows <= 1024 ? kNormRows : 1;
    const dim3 grid((whole + rows - 1) / rows), block(per_row * rows);
    const long long stride = (long long)M * d;
#define IC_NORM_PARTS(V, R) hipLaunchKernelGGL((norm_parts_kernel<V, R>), grid, block, 0, stream, x, y, n_slices, stride, alpha, w, out, (unsigned char*)parts, M, d, eps)
    if (rows > 1) IC_NORM_PARTS(1, kNormRows);
    else if (vpt == 1) IC_NORM_PARTS(1, 1);
    else if (vpt == 2) IC_NORM_PARTS(2, 1);
    else if (vpt == 3) IC_NORM_PARTS(3, 1);
    else IC_NORM_PARTS(4, 1);
#undef IC_NORM_PARTS
    return ic_launch_status();
}

// act (float32 [M, di]) = up * silu(gate) of gate_up [M, 2 di] (gate, then up), in three parts at `parts` too; di a multiple of 32, all 16-byte aligned.
IC_EXPORT int ic_swiglu_parts_f32(const float* gate_up, float* act, void* parts, int M, int di, hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!gate_up || !act || !parts || di < 32 || di % 32 || M > (1 << 26) || !aligned16(gate_up) || !aligned16(act) || !aligned16(parts)) return IC_ERR_ARG;
    const long long waves = (long long)((M + 15) / 16) * (di / 32);
    if (waves >= (1LL << 30)) return IC_ERR_ARG;
    hipLaunchKernelGGL(swiglu_parts_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, stream, gate_up, act, M, di, (uint4*)parts);
    return ic_launch_status();
}
