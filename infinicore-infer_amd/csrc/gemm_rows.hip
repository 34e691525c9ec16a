// C = alpha * A[M, K] W[N, K]^T for up to 8 rows in bfloat16 with an epilogue (gate/up with the gated unit, QKV with rotary and
// cache write, the projections into the residual stream): weights from memory straight into the operands of the matrix cores.
//
// A wave's load covers 8 weight rows x 128 bytes, whole cache lines, and what it brings is an operand of
// v_mfma_f32_16x16x32_bf16 as it is: lane l holds row l % 8, and 16 bytes of it number l / 16 + 4 (l / 8 % 2).  Operand row i < 8
// is then weight row i with the first 32 k of the line, operand row i >= 8 weight row i - 8 with the second 32.  The token
// operand is loaded the same way (column j: token j % 8, the line's half j / 8), so of D[i][j] the quarters i < 8, j < 8 and
// i >= 8, j >= 8 are the two halves' sums and the other two quarters are dropped: half the matrix work, of which there is plenty,
// for no pass of the weights through LDS and loads that can all be in flight at once.
#include "gemm_rows.h"

namespace {

typedef __bf16 gr_v8b __attribute__((ext_vector_type(8)));
typedef float gr_v4f __attribute__((ext_vector_type(4)));
typedef const void __attribute__((address_space(1)))* gr_gptr;
typedef void __attribute__((address_space(3)))* gr_lptr;

__device__ __forceinline__ gr_v8b gr_op(const uint4& v) { return __builtin_bit_cast(gr_v8b, v); }

// floats of LDS: the waves' halves of the results, the waves' sums of squares, with STAGE the token rows (8 KB per 512 k)
constexpr int gr_lds_floats(int groups, int waves) { return 2 * waves * groups * 64 + 8 * waves; }

// RG: groups of 8 weight rows per block (EPI 1 and 2: half of them gate rows and half up rows, or pairs that rotate together).
// UL: lines of a register stage.  STAGE: the token rows go through LDS once per block instead of to every wave by itself.
template <int EPI, int RG, int UL, int WV, bool STAGE>
__global__ void __launch_bounds__(64 * WV)
gemm_rows_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W, bf16* __restrict__ C, int M, int N, int K, int lda,
                 int ldw, int ldc, float alpha, RopeEpilogue rope, NormFuse nf, int cols) {
    constexpr bool PAIRED = EPI == 1 || EPI == 2;
    static_assert(!PAIRED || RG % 2 == 0, "gate and up rows, and rows that rotate together, come in pairs of groups");
    constexpr int OUT = RG * 64;                             // results of a block: [group][token][row]
    static_assert((PAIRED ? OUT / 2 : OUT) <= 64 * WV, "a thread owns at most one result");
    extern __shared__ __align__(16) float gr_smem[];
    float* const red = gr_smem;                              // [2 waves][OUT]
    float* const ssum = gr_smem + 2 * WV * OUT;              // [waves][8]
    unsigned char* const rows = reinterpret_cast<unsigned char*>(gr_smem + gr_lds_floats(RG, WV));       // [K / 64][8 tokens][128 bytes]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r8 = lane & 7, hi = (lane >> 3) & 1, kq = lane >> 4;
    const int NO = EPI == 1 ? N / 2 : N, lines = K >> 6;

    if constexpr (STAGE) {
        // line l of the 8 token rows (rows beyond M repeat the last one): lane i brings 16 bytes, number i % 8, of token i / 8
        const int m = (lane >> 3) < M ? (lane >> 3) : M - 1;
        const uint16_t* src = A + (size_t)m * lda + 8 * (lane & 7);
        for (int l = wave; l < lines; l += WV)
            __builtin_amdgcn_global_load_lds((gr_gptr)(src + 64 * l), (gr_lptr)(rows + 1024 * l), 16, 0, 0);
    }

    const uint16_t* wp[RG];
    const int col8 = 8 * (kq + 4 * hi);
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        int row, last;
        if constexpr (EPI == 1) {
            const int first = (int)blockIdx.x * cols + 8 * (g % (RG / 2)), up = (g / (RG / 2)) * NO;
            row = first + r8 + up;
            last = NO - 1 + up;
        } else if constexpr (EPI == 2) {
            const int pair = (int)blockIdx.x * (RG / 2) + (g >> 1), per_head = rope.dh >> 4;
            const int head = pair / per_head, j = 8 * (pair - head * per_head);
            row = head * rope.dh + r8 + (head < rope.nh + rope.nkvh ? j + (g & 1) * (rope.dh >> 1) : 2 * j + 8 * (g & 1));
            last = N - 1;
        } else {
            row = (int)blockIdx.x * cols + 8 * g + r8;
            last = ((int)blockIdx.x + 1) * cols - 1;
            last = last < N - 1 ? last : N - 1;
        }
        wp[g] = W + (size_t)(row < last ? row : last) * ldw + col8;
    }
    const uint16_t* const ap = A + (size_t)(r8 < M ? r8 : M - 1) * lda + col8;

    // what the epilogue needs is asked for first and used last
    constexpr int PV = (kMaxSumParts + 8 * WV - 1) / (8 * WV);          // column blocks a thread sums
    float pv[PV];
    if (nf.ss_in) {
#pragma unroll
        for (int i = 0; i < PV; ++i) {
            const int p = (tid >> 3) + i * 8 * WV;
            pv[i] = p < nf.n_parts_in ? nf.ss_in[p * 16 + (tid & 7)] : 0.f;
        }
    }
    // this thread's result: group (or pair of groups) og, token om, row oi of the group
    const int oi = tid & 7, om = (tid >> 3) & 7, og = tid >> 6;
    const bool owner = tid < (PAIRED ? OUT / 2 : OUT) && om < M;
    float e0 = 0.f, e1 = 0.f;
    int on = 0, slot = -1, pos = 0, head = 0, hj = 0;
    bool mine_ok = owner;
    if constexpr (EPI == 2) {
        const int pair = (int)blockIdx.x * (RG / 2) + og, per_head = rope.dh >> 4;
        head = pair / per_head;
        hj = 8 * (pair - head * per_head);
        mine_ok = owner && head < rope.nh + 2 * rope.nkvh;
        if (mine_ok) { slot = rope.slots[om]; pos = rope.positions[om]; }
    } else {
        on = (int)blockIdx.x * cols + 8 * og + oi;
        mine_ok = owner && 8 * og + oi < cols && on < NO;
        if (EPI == 3 && mine_ok) { e0 = nf.x[(size_t)om * nf.ldx + on]; e1 = nf.g[on]; }
    }

    uint4 wr[2][UL][RG], ar[2][UL];
    // a stage: lines l0, l0 + WV, ..; of the first n of them (the others repeat the first: a load is never conditional)
    auto issue = [&](int l0, int n, uint4 (&w)[UL][RG], uint4 (&a)[UL]) {
#pragma unroll
        for (int u = 0; u < UL; ++u) {
            const int l = u < n ? l0 + u * WV : l0;
#pragma unroll
            for (int g = 0; g < RG; ++g) w[u][g] = load_stream16(wp[g] + 64 * l);
            if constexpr (!STAGE) a[u] = *reinterpret_cast<const uint4*>(ap + 64 * l);
        }
    };
    gr_v4f acc[RG];
#pragma unroll
    for (int g = 0; g < RG; ++g) acc[g] = gr_v4f{0.f, 0.f, 0.f, 0.f};
    auto use = [&](int l0, int n, const uint4 (&w)[UL][RG], uint4 (&a)[UL]) {
#pragma unroll
        for (int u = 0; u < UL; ++u) {
            if (u < n) {                                     // (uniform in the wave)
                if constexpr (STAGE) a[u] = *reinterpret_cast<const uint4*>(rows + 1024 * (l0 + u * WV) + 128 * r8 + 16 * (kq + 4 * hi));
#pragma unroll
                for (int g = 0; g < RG; ++g) acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(gr_op(w[u][g]), gr_op(a[u]), acc[g], 0, 0, 0);
            }
        }
    };
    int left = (lines - wave + WV - 1) / WV, l = wave;       // lines of this wave
    if (left > 0) issue(l, left, wr[0], ar[0]);
    if constexpr (EPI == 2) {
        if (mine_ok && head < rope.nh + rope.nkvh) {
            const size_t at = (size_t)pos * (rope.dh >> 1) + hj + oi;
            e0 = rope.cos_t[at];
            e1 = rope.sin_t[at];
        }
    }
    if constexpr (STAGE) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // this wave's token lines have reached LDS (and its first weights are here)
        __syncthreads();                                     // everybody's have
    }
    if (left > 0) {
        while (true) {
            if (left <= UL) { use(l, left, wr[0], ar[0]); break; }
            issue(l + UL * WV, left - UL, wr[1], ar[1]);
            use(l, UL, wr[0], ar[0]);
            l += UL * WV; left -= UL;
            if (left <= UL) { use(l, left, wr[1], ar[1]); break; }
            issue(l + UL * WV, left - UL, wr[0], ar[0]);
            use(l, UL, wr[1], ar[1]);
            l += UL * WV; left -= UL;
        }
    }

    // D[i = 4 kq + e][j = l % 16]: the two quarters that count (hi == kq / 2)
    if (hi == (kq >> 1)) {
#pragma unroll
        for (int g = 0; g < RG; ++g) *reinterpret_cast<gr_v4f*>(red + (2 * wave + hi) * OUT + g * 64 + 8 * r8 + 4 * (kq & 1)) = acc[g];
    }
    if (nf.ss_in) {
        float t = 0.f;
#pragma unroll
        for (int i = 0; i < PV; ++i) t += pv[i];
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) t += __shfl_xor(t, o, kWave);
        if (lane < 8) ssum[wave * 8 + lane] = t;
    }
    __syncthreads();
    float f = alpha;
    if (nf.ss_in) {
        float t = 0.f;
#pragma unroll
        for (int w = 0; w < WV; ++w) t += ssum[w * 8 + om];
        f *= rsqrtf(t * nf.inv_width + nf.eps);
    }
    // a projection's result, rounded to its type first, as when it is stored
    auto result = [&](int at) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < 2 * WV; ++w) v += red[w * OUT + at];
        return to_f32(from_f32<bf16>(f * v));
    };
    if constexpr (EPI == 1) {
        if (!mine_ok) return;
        const float g = result(tid), u = result(tid + OUT / 2);
        C[(size_t)om * ldc + on] = from_f32<bf16>(nf.glu_limit > 0.f ? glu_clamped_f(g, u, nf.glu_limit, nf.glu_slope) : silu_mul_fast(g, u));
    } else if constexpr (EPI == 2) {
        if (!mine_ok || (head >= rope.nh && slot < 0)) return;
        const float v0 = result(2 * og * 64 + (tid & 63)), v1 = result((2 * og + 1) * 64 + (tid & 63));
        const int page = slot >= 0 ? slot / rope.page_size : 0, off = slot >= 0 ? slot - page * rope.page_size : 0;
        if (head >= rope.nh + rope.nkvh) {
            bf16* dst = (bf16*)rope.vcache + (((size_t)page * rope.nkvh + (head - rope.nh - rope.nkvh)) * rope.page_size + off) * rope.dh + 2 * hj + oi;
            dst[0] = from_f32<bf16>(v0);
            dst[8] = from_f32<bf16>(v1);
            return;
        }
        bf16* dst = head < rope.nh ? C + (size_t)om * ldc + (size_t)head * rope.dh
                                   : (bf16*)rope.kcache + (((size_t)page * rope.nkvh + (head - rope.nh)) * rope.page_size + off) * rope.dh;
        dst[hj + oi] = from_f32<bf16>(v0 * e0 - v1 * e1);
        dst[hj + (rope.dh >> 1) + oi] = from_f32<bf16>(v0 * e1 + v1 * e0);
    } else {
        float ss = 0.f;
        if (mine_ok) {
            const float h = e0 + nf.rscale * result(tid);
            nf.x[(size_t)om * nf.ldx + on] = h;
            C[(size_t)om * ldc + on] = from_f32<bf16>(h * e1);
            ss = h * h;
        }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) ss += __shfl_xor(ss, o, kWave);
        if constexpr (RG == 1) {
            if (tid < OUT && oi == 0) {
                nf.ss_out[blockIdx.x * 16 + om] = ss;
                nf.ss_out[blockIdx.x * 16 + 8 + om] = 0.f;   // token rows that this kernel does not take
            }
        } else {
            __syncthreads();                                 // the results have been read
            if (tid < OUT && oi == 0) red[og * 8 + om] = ss;
            __syncthreads();
            if (tid < 16) {
                float t = 0.f;
                if (tid < 8)
#pragma unroll
                    for (int g = 0; g < RG; ++g) t += red[g * 8 + tid];
                nf.ss_out[blockIdx.x * 16 + tid] = t;
            }
        }
    }
}

template <int EPI, int RG, int UL, int WV, bool STAGE>
bool gr_launch(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha, const RopeEpilogue& rope,
               const NormFuse& nf, int blocks, int cols, hipStream_t stream) {
    const size_t lds = gr_lds_floats(RG, WV) * sizeof(float) + (STAGE ? (size_t)K * 16 : 0);
    if (lds > 160 * 1024) return false;
    if (lds > 64 * 1024) {
        static bool raised[64] = {};                         // per device: the kernel may use more than 64 KB of LDS
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return false;
        if (!raised[dev]) {
            if (hipFuncSetAttribute((const void*)gemm_rows_kernel<EPI, RG, UL, WV, STAGE>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            raised[dev] = true;
        }
    }
    hipLaunchKernelGGL((gemm_rows_kernel<EPI, RG, UL, WV, STAGE>), dim3(blocks), dim3(64 * WV), lds, stream, (const uint16_t*)A,
                       (const uint16_t*)W, (bf16*)C, M, N, K, lda, ldw, ldc, alpha, rope, nf, cols);
    return true;
}

}  // namespace

// What it takes and why, against the kernel of gemm.hip whose weights pass through LDS (chains of recorded launches over weights that
// are not in the caches; us, that kernel / this one at 1, 4 and 8 rows):
//   1B shape (1,536 wide):  QKV 5.8 / 4.9, 5.9 / 5.1, 6.4 / 5.2;  O 4.7 / 3.9, 4.9 / 4.3, 5.1 / 4.1;
//                           gate/up 7.0 / 6.5, 7.0 / 6.5, 7.5 / 6.8;  down 5.7 / 4.7, 6.0 / 5.3, 6.7 / 5.6
//   2B shape (2,304 wide):  QKV 8.4 / 8.2, 8.5 / 8.3, 8.9 / 9.0;  O 5.3 / 4.8, 5.5 / 5.2, 6.1 / 5.5;
//                           gate/up 11.9 / 10.8, 12.1 / 10.8, 12.2 / 10.9;  down 7.5 / 7.4, 7.7 / -, 8.6 / 8.6
//   8B shape (4,096 wide):  QKV 11.5 / -, 12.2 / 12.0, 12.5 / 11.9;  O 8.1 / 7.9, 8.4 / 8.1, 8.7 / 8.7;  gate/up 43.1 / 41.8, 43.2 / 41.4, 43.5 / 42.4
// A kernel that only loads these weights takes 2.3 (O of the 1B shape) to 9.9 us (gate/up of the 2B shape), an empty one 1.7.
// Not taken: 9 rows and more (a second set of token operands; 16 rows were slower throughout), rows of 16 KB and more (8B shape's down
// projection 23.8 / 24.6 .. 27.8: there a wave's one stretch of every row counts), and 1..3 rows of QKV in fewer blocks than three
// quarters of the units.  The token rows go through LDS from 5 rows on (each wave fetching them for itself reads as many bytes of
// tokens as of weights), except where a block's groups are many enough to share them.
bool gemm_rows_launch(int epi, const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, float alpha,
                      const RopeEpilogue& rope, const NormFuse& nf, int blocks, hipStream_t stream) {
    if (M < 1 || M > 8 || K < 64 || K % 64 || K >= 8192 || lda % 8 || ldw % 8 || ((((uintptr_t)A) | (uintptr_t)W) & 15)) return false;
    constexpr int kUnits = 256;                              // compute units that the splits below are made for
    const bool stage = M > 4;
#define GR_GO(EPI, RG, UL, WV, STAGE, BLOCKS, COLS) \
    return gr_launch<EPI, RG, UL, WV, STAGE>(A, W, C, M, N, K, lda, ldw, ldc, alpha, rope, nf, BLOCKS, COLS, stream)
    if (epi == 1) {
        // 1, 2 or 3 groups of gate rows a block when one round of blocks then takes them all, else 2
        const int groups = (N / 2 + 7) / 8, per = (groups + kUnits - 1) / kUnits;
        if (per == 1) GR_GO(1, 2, 2, 8, false, groups, 8);
        if (per == 3) GR_GO(1, 6, 1, 8, false, (groups + 2) / 3, 24);
        GR_GO(1, 4, 1, 8, false, (groups + 1) / 2, 16);
    }
    if (epi == 2) {
        const int pairs = (rope.nh + 2 * rope.nkvh) * (rope.dh / 16), two = (pairs + 1) / 2;
        if (pairs <= kUnits) { if (stage) GR_GO(2, 2, 2, 12, true, pairs, 0); GR_GO(2, 2, 2, 12, false, pairs, 0); }
        if (M < 4 && 4 * two < 3 * kUnits) return false;
        if (stage) GR_GO(2, 4, 1, 16, true, two, 0);
        GR_GO(2, 4, 1, 12, false, two, 0);
    }
    if (epi == 3) {
        const int cols = blocks > 0 ? (N + blocks - 1) / blocks : 0;       // as gemm.hip deals them: one block a unit, or 16 columns
        if (cols < 1 || cols > 16) return false;
        if (K > 4608 && M > 2 && M <= 4) return false;       // (2B shape's down projection: 7.6, 7.8 there, 7.8, 8.1 here)
        if (cols <= 8) { if (stage) GR_GO(3, 1, 4, 8, true, blocks, cols); GR_GO(3, 1, 4, 8, false, blocks, cols); }
        if (cols == 16) GR_GO(3, 2, 2, 16, false, blocks, cols);
        if (stage && K > 4608) GR_GO(3, 2, 2, 12, true, blocks, cols);
        if (stage) GR_GO(3, 2, 2, 8, true, blocks, cols);
        GR_GO(3, 2, 2, 8, false, blocks, cols);
    }
#undef GR_GO
    return false;
}
