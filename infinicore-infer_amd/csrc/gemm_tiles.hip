// C[M, N] = A[M, K] * W[N, K]^T for many rows M (prompts and mixed steps): bfloat16 operands on the matrix cores, float32
// accumulation, the result's next operation in the epilogue.
//
// A block of WM x WN x WK waves owns a tile of BM rows of A by BN rows of W.  Both operands go from memory straight into LDS
// (global_load_lds_dwordx4, 1 KB an instruction and wave), STAGES stages of 64 k deep: rows of 128 bytes without padding, the
// 16-byte chunk c of row r at position c ^ (r / 2 % 8), which each lane arranges by what it fetches, so that the operand reads of
// 16 rows cover the 64 banks once.  A wave holds TM x TN results (TM = BM / WM, TN = BN / WN) in registers and walks every WK-th
// k-step of 32; with WK > 1 the waves of a tile meet in LDS at the end.
//
// The walk over K: the operands of a k-step are read from LDS while the previous step is multiplied.  Before the last step of a
// stage is multiplied a wave waits for its own loads of the next stage and for its reads of this one, then all waves meet: after
// that barrier the next stage is whole and this one is free, and the loads of the stage STAGES further on go into it.  So loads
// have STAGES - 1 stages of products to arrive, and there is one barrier a stage.  The loads are written as inline assembly: the
// compiler, which cannot see which LDS bytes such a load writes, otherwise waits for all of them before every operand read.  They
// have no register results, so nothing but LDS is written while they are in flight.
//
// What bounds it.  Few tiles (up to one a compute unit): a stage's products at the matrix cores' rate plus its barrier and what the loads hold up the
// products: 256 x 256 0.96 us a stage (0.87 with products alone), 128 x 128 0.30 (0.23), and about 4 us for launch, first
// loads and the way out.  128 x 128 tiles take all of a unit's 64 bytes a cycle from L2 for their loads, 256 x 256 half of it, hence the large
// tiles where there are rows and columns enough.  The whole chip busy for long: its power, the clock gives way (256 x 256: 1.43 us a stage in gate/up of
// 16,384 x 32,768 x 4,096, 1.68 in 16,384 x 4,096 x 16,384).
// Large tiles take four waves of up to 512 registers a block: eight waves of half the size read 1.5 times as much from LDS
// (256 x 256: 1.07 us a stage).  v_mfma_f32_32x32x16_bf16 instead of 16x16x32 is no faster (0.96 and 0.97).
//
// 16x16x32 layout (lane l): A[i = l%16][k = 8(l/16)..+7], B[k = 8(l/16)..+7][j = l%16], D[i = 4(l/16) + e][j = l%16], e = 0..3;
// i are weight rows here and j token rows, so a lane holds four neighbouring columns of one row of C.
#include "common.h"
#include "infinicore_infer_variants.h"
#include <type_traits>
#include <utility>

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

struct TilesArgs {
    const uint16_t* A;
    const uint16_t* W;
    uint16_t* C;
    int M, N, K, lda, ldw, ldc;   // N: rows of W
    int tiles_m, tiles_n;         // the grid: tiles_m * tiles_n blocks
    int group_m;                  // row tiles that are walked together
    // EPI_ROPE: W = [q heads; k heads; v heads], rows of 2 half = 2 << half_log
    const int* positions;
    const int* slots;
    const float* cos_t;           // [positions, half]
    const float* sin_t;
    uint16_t* kcache;             // [pages, kv heads, page size, 2 half]
    uint16_t* vcache;
    int nh, nkvh, half_log, page_size;
};

// What follows the product.  SWIGLU and ROPE are about pairs of columns (gate and up of one column; a head's entries j and j + half): C counts in
// pairs, and a wave's TN weight rows are the first members of TN / 2 neighbouring pairs, then their second ones, so that a lane has both.
enum { EPI_BF16 = 0, EPI_SWIGLU = 1, EPI_ROPE = 2 };

// 16 bytes a lane from base + off (bytes; base the same for the wave) to LDS at lds + plus + 16 * lane.
template <int PLUS> __device__ __forceinline__ void load_to_lds(unsigned lds, unsigned off, const char* base) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base), "i"(PLUS) : "memory", "scc");
}
// waits until at most N of this wave's loads are on their way and all its LDS reads are done
template <int N> __device__ __forceinline__ void wait_loads() {
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (0 << 8));
}
constexpr int min_of(int a, int b) { return a < b ? a : b; }
// f(0), f(1), .. f(N - 1), each with its number as a type
template <typename F, int... Is> __device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void each(F&& f) { each_of(f, std::make_integer_sequence<int, N>{}); }

// acc += w a.  OWN: with 256 accumulators a lane, all of the second half of its 512 registers, the compiler's own product copies them from product to
// product (192 copies a stage; with ROPE's way out, which needs more registers, in all tiles of 32 accumulators and more); written as assembly, with
// an operand that is read and written, it does not.  The compiler does not know such a product for one and adds no wait before an instruction that
// reads its result: LAST, on the last product of a k-step, waits here (11 wait states after eight passes), so that whatever follows the k-step may read
// any accumulator.  settled() ties the accumulators to a place between the volatile products: what writes or reads them stays on its side of it.
template <bool OWN, bool LAST> __device__ __forceinline__ void product(v4f& acc, const v8b& w, const v8b& a) {
    if constexpr (!OWN) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, acc, 0, 0, 0);
    else if constexpr (LAST) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\ts_nop 15" : "+a"(acc) : "v"(w), "v"(a));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(a));
}

template <bool OWN, int N, int M> __device__ __forceinline__ void settled(v4f (&acc)[N][M]) {
    if constexpr (OWN) {
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int m = 0; m < M; ++m) asm volatile("" : "+a"(acc[n][m]));
        asm volatile("s_nop 7");
    }
}

template <int BM_, int BN_, int WM_, int WN_, int WK_, int STAGES_> struct Tile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, WK = WK_, STAGES = STAGES_;
    static constexpr int WAVES = WM * WN * WK, TM = BM / WM, TN = BN / WN, MT = TM / 16, NT = TN / 16;
    static constexpr int STEPS = 2 / WK;                           // k-steps of a stage that a wave multiplies
    static constexpr int STAGE_BYTES = (BM + BN) * 128;
    static constexpr int LOADS_A = BM / 8 / WAVES, LOADS = LOADS_A + BN / 8 / WAVES;    // of 1 KB, a wave and stage
    static constexpr int SUM_BYTES = BM * BN * 4 * (WK - 1);
    static constexpr int LDS_BYTES = STAGES * STAGE_BYTES > SUM_BYTES ? STAGES * STAGE_BYTES : SUM_BYTES;
    // (with ROPE 256 accumulators a lane leave too few registers for the way out: 2,048 x 6,912 x 2,304 71 us, product and rotary's own kernel 67)
    static constexpr bool takes(int epi) { return epi == EPI_BF16 || (NT % 2 == 0 && !(epi == EPI_ROPE && TM * TN / 64 > 192)); }
    static constexpr bool own_product(int epi) { return TM * TN / 64 > 192 || (epi == EPI_ROPE && STEPS > 1); }
    static constexpr int BLOCKS_PER_CU = LDS_BYTES <= 80 * 1024 ? 2 : 1;
    static_assert(BM % (16 * WM) == 0 && BN % (16 * WN) == 0, "whole matrix tiles");
    static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "every wave loads as much");
    static_assert(STEPS == 1 || STEPS == 2, "a stage is two k-steps");
    static_assert((WAVES == 4) && MT % WK == 0 && LDS_BYTES <= 160 * 1024 && LOADS * (STAGES - 1) < 64, "limits");
};

template <typename T, int EPI>
__global__ void __launch_bounds__(T::WAVES * 64, T::BLOCKS_PER_CU) gemm_tiles_kernel(TilesArgs a) {
    constexpr int BM = T::BM, BN = T::BN, WN = T::WN, WK = T::WK, STAGES = T::STAGES, WAVES = T::WAVES;
    constexpr int TM = T::TM, TN = T::TN, MT = T::MT, NT = T::NT, STEPS = T::STEPS, LOADS = T::LOADS, LOADS_A = T::LOADS_A;
    static_assert(T::takes(EPI), "a wave holds both of a pair");
    __shared__ __attribute__((aligned(1024))) unsigned char lds[T::LDS_BYTES];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kq = lane >> 4;
    const int wk = wave % WK, wn = wave / WK % WN, wm = wave / (WK * WN);

    // Which tile: blocks go to the 8 XCDs in turn, so block b is the (b / 8)-th of XCD b % 8, and every XCD takes one run of tiles
    // (its L2 then holds few rows of W and A); a run goes down group_m row tiles, then to the next columns.
    const int total = a.tiles_m * a.tiles_n;
    const int xcd = blockIdx.x & 7, nth = blockIdx.x >> 3;
    const int t = xcd * (total >> 3) + min(xcd, total & 7) + nth;
    const int group = t / (a.group_m * a.tiles_n), first_m = group * a.group_m;
    const int gm = min(a.group_m, a.tiles_m - first_m), in_group = t - group * a.group_m * a.tiles_n;
    const int bn = in_group / gm, bm = first_m + in_group - bn * gm;
    const int m0 = bm * BM;
    constexpr bool PAIRS = EPI != EPI_BF16;
    const int NO = PAIRS ? a.N / 2 : a.N;                          // columns of C, or pairs
    constexpr int BNO = PAIRS ? BN / 2 : BN;
    const int n0 = bn * BNO;

    const int n_stages = a.K / 64;

    // What this lane fetches: byte offsets from the tile's first row of A, or from W (rows beyond the matrix repeat the last one)
    const char* base_a = (const char*)(a.A + (size_t)m0 * a.lda);
    const char* base_w = (const char*)(a.W + (PAIRS ? (size_t)0 : (size_t)n0 * a.ldw));
    unsigned off[LOADS];
    each<LOADS>([&](auto at) {
        constexpr int I = decltype(at)::value;
        const int row = 8 * (wave + WAVES * (I < LOADS_A ? I : I - LOADS_A)) + (lane >> 3);
        const unsigned chunk = 16 * ((lane & 7) ^ ((row >> 1) & 7));
        if constexpr (I < LOADS_A) {
            off[I] = (unsigned)min(row, a.M - 1 - m0) * (unsigned)(a.lda * 2) + chunk;
        } else if constexpr (PAIRS) {
            const int x = row % TN, pair = min(n0 + row / TN * (TN / 2) + x % (TN / 2), NO - 1);
            const int first = EPI == EPI_ROPE ? pair + ((pair >> a.half_log) << a.half_log) : pair;
            const int apart = EPI == EPI_ROPE ? 1 << a.half_log : NO;
            off[I] = (unsigned)(first + (x >= TN / 2 ? apart : 0)) * (unsigned)(a.ldw * 2) + chunk;
        } else {
            off[I] = (unsigned)min(row, a.N - 1 - n0) * (unsigned)(a.ldw * 2) + chunk;
        }
    });
    // this wave's I-th load of a stage: at_a, at_w are the stage's bases, into the buffer at LDS address `into` (of this wave's first chunk)
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds + wave * 1024;
    auto fetch = [&](auto at, const char* at_a, const char* at_w, unsigned into) {
        constexpr int I = decltype(at)::value;
        if constexpr (I < LOADS_A) load_to_lds<I * WAVES * 1024>(into, off[I], at_a);
        else load_to_lds<BM * 128 + (I - LOADS_A) * WAVES * 1024>(into, off[I], at_w);
    };

    constexpr int SH = MT / WK;                                    // row tiles of C this wave writes: SH from the wk-th run on
    const int row0 = m0 + wm * TM + wk * (16 * SH);
    // ROPE: positions and cache slots of this lane's rows, asked for now and used last
    int pos[SH], slot[SH];
    if constexpr (EPI == EPI_ROPE) {
#pragma unroll
        for (int j = 0; j < SH; ++j) {
            const int row = min(row0 + 16 * j + r, a.M - 1);
            pos[j] = a.positions[row];
            slot[j] = a.slots[row];
        }
    }

    v4f acc[NT][MT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = v4f{0.f, 0.f, 0.f, 0.f};
    settled<T::own_product(EPI)>(acc);                             // (the compiler waits neither between these writes and the first products)

    // operand registers of two k-steps: one is multiplied while the other is read
    v8b fa[2][MT], fw[2][NT];
    const unsigned char* const pa = lds + (wm * TM + r) * 128;
    const unsigned char* const pw = lds + (BM + wn * TN + r) * 128;
    const int sw = (r >> 1) & 7;
    // byte of a row where step `step` (of the wave's STEPS in a stage) has this lane's eight k
    auto place = [&](int step) { return 16 * ((4 * (step * WK + wk) + kq) ^ sw); };

    // The loads of stage s + STAGES go into the buffer of stage s from that stage's barrier on: with more than two stages SPREAD of them in each
    // k-step up to the next barrier, so that they do not queue up behind one another (a 1 KB load takes the unit 16 cycles, and a wave that
    // waits to issue one issues no products: 128 x 128 tiles 0.40 -> 0.30 us a stage); with two the last ones would have to arrive too soon.
    constexpr int SPREAD = STAGES > 2 ? (LOADS + STEPS - 1) / STEPS : LOADS;
    // the first stages, the last of them without what the first stage's steps load
    each<STAGES>([&](auto sc) {
        constexpr int S = decltype(sc)::value;
        const int from = 128 * min(S, n_stages - 1);
        each<S + 1 < STAGES ? LOADS : SPREAD>([&](auto i) { fetch(i, base_a + from, base_w + from, lds0 + S * T::STAGE_BYTES); });
    });
    wait_loads<LOADS * (STAGES - 2) + SPREAD>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) fw[0][nt] = *reinterpret_cast<const v8b*>(pw + place(0) + nt * 2048);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) fa[0][mt] = *reinterpret_cast<const v8b*>(pa + place(0) + mt * 2048);

    // One k-step: the registers CUR are multiplied while the others are read (step `step` of the stage in `buf`) and this wave's loads
    // FROM .. TO - 1 of the stage at at_a, at_w go out.  The reads are dealt over the first three quarters of the products, the loads over all of
    // them: left to itself the scheduler moves them all to the end, where the next step waits for them.
    auto step_of = [&](auto curc, auto fromc, auto toc, int buf, int step, const char* at_a, const char* at_w, unsigned into) {
        constexpr int CUR = decltype(curc)::value, P = MT * NT, R = NT + MT, L0 = decltype(fromc)::value, L = decltype(toc)::value - L0;
        const unsigned char* const qa = pa + buf * T::STAGE_BYTES + place(step);
        const unsigned char* const qw = pw + buf * T::STAGE_BYTES + place(step);
        each<P>([&](auto at) {
            constexpr int I = decltype(at)::value;
            constexpr int R0 = I == 0 ? 0 : min_of(R, 4 * (I - 1) * R / (3 * P) + 1), R1 = min_of(R, 4 * I * R / (3 * P) + 1);
            constexpr int F0 = I == 0 || L == 0 ? 0 : min_of(L, (I - 1) * L / P + 1), F1 = L == 0 ? 0 : min_of(L, I * L / P + 1);
            each<R1 - R0>([&](auto k) {
                constexpr int O = R0 + decltype(k)::value;
                if constexpr (O < NT) fw[CUR ^ 1][O] = *reinterpret_cast<const v8b*>(qw + O * 2048);
                else fa[CUR ^ 1][O - NT] = *reinterpret_cast<const v8b*>(qa + (O - NT) * 2048);
            });
            each<F1 - F0>([&](auto k) { fetch(std::integral_constant<int, L0 + F0 + decltype(k)::value>{}, at_a, at_w, into); });
            if constexpr (R1 > R0 || F1 > F0) __builtin_amdgcn_sched_barrier(0);
            product<T::own_product(EPI), I + 1 == P>(acc[I / MT][I % MT], fw[CUR][I / MT], fa[CUR][I % MT]);
        });
        __builtin_amdgcn_sched_barrier(0);
    };
    // where they come from: beyond the last stage that one is loaded again (and read by nobody)
    const char *ahead_a = base_a + 128 * min(STAGES - 1, n_stages - 1), *ahead_w = base_w + 128 * min(STAGES - 1, n_stages - 1);
    auto whole_stage = [&](int s, int buf, auto cur0) {            // cur0: which operand registers hold its first step
        const int next = buf + 1 == STAGES ? 0 : buf + 1, before = buf == 0 ? STAGES - 1 : buf - 1;
        each<STEPS>([&](auto pc) {
            constexpr int P = decltype(pc)::value;
            using Cur = std::integral_constant<int, (decltype(cur0)::value + P) & 1>;
            if constexpr (P + 1 < STEPS) {
                step_of(Cur{}, std::integral_constant<int, SPREAD>{}, std::integral_constant<int, LOADS>{}, buf, P + 1, ahead_a, ahead_w,
                        lds0 + before * T::STAGE_BYTES);
            } else {
                wait_loads<LOADS * (STAGES - 2)>();                // under way: stages s + 1 .. s + STAGES - 1
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                const int on = s + STAGES < n_stages ? 128 : 0;
                ahead_a += on;
                ahead_w += on;
                step_of(Cur{}, std::integral_constant<int, 0>{}, std::integral_constant<int, SPREAD>{}, next, 0, ahead_a, ahead_w,
                        lds0 + buf * T::STAGE_BYTES);
            }
        });
        return next;
    };
    int s = 0, buf = 0;
    if constexpr (STEPS == 1) {                                    // two stages a round, so that the operand registers are named by constants
        for (; s + 1 < n_stages; s += 2) {
            buf = whole_stage(s, buf, std::integral_constant<int, 0>{});
            buf = whole_stage(s + 1, buf, std::integral_constant<int, 1>{});
        }
        if (s < n_stages) whole_stage(s, buf, std::integral_constant<int, 0>{});
    } else {
        for (; s < n_stages; ++s) buf = whole_stage(s, buf, std::integral_constant<int, 0>{});
    }
    settled<T::own_product(EPI)>(acc);
    wait_loads<0>();
    __syncthreads();                                               // LDS is free

    if constexpr (WK > 1) {
        // the WK waves of the same results add up, each its own run of rows
        float* const red = reinterpret_cast<float*>(lds) + (size_t)(wm * WN + wn) * (WK * (WK - 1) * SH * NT * 256);
        auto cell = [&](int whose, int src, int j, int nt) {
            return reinterpret_cast<v4f*>(red + ((((whose * (WK - 1) + src) * SH + j) * NT + nt) * 64 + lane) * 4);
        };
#pragma unroll
        for (int o = 0; o < WK; ++o)                               // o: whose run
            if (o != wk) {
#pragma unroll
                for (int j = 0; j < SH; ++j)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) *cell(o, wk < o ? wk : wk - 1, j, nt) = acc[nt][o * SH + j];
            }
        __syncthreads();
#pragma unroll
        for (int o = 1; o < WK; ++o)
            if (o == wk) {
#pragma unroll
                for (int j = 0; j < SH; ++j)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) acc[nt][j] = acc[nt][o * SH + j];
            }
#pragma unroll
        for (int src = 0; src < WK - 1; ++src)
#pragma unroll
            for (int j = 0; j < SH; ++j)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) acc[nt][j] += *cell(wk, src, j, nt);
        __syncthreads();
    }
    constexpr int ONT = PAIRS ? NT / 2 : NT;                       // column tiles of C, or of pairs
    const int c0 = n0 + wn * (ONT * 16);

    // 16 rows at a time through LDS of the wave's own, so that whole lines are stored
    constexpr int PARTS = EPI == EPI_ROPE ? 2 : 1;                 // of a row: a pair's first members, then its second ones
    constexpr int ROW = PARTS * ONT * 32 + 16, PER_ROW = PARTS * ONT * 2;      // bytes of a row in LDS; 16-byte chunks of a row
    constexpr int CELLS = EPI == EPI_ROPE ? SH * 128 : 0;
    unsigned char* const mine = lds + wave * (16 * ROW + CELLS);
    long long* const cell_of = reinterpret_cast<long long*>(mine + 16 * ROW);  // where a row's kv head 0 lies in the cache, -1: nowhere
    static_assert(WAVES * (16 * ROW + CELLS) <= T::LDS_BYTES, "room for the rows");
    if constexpr (EPI == EPI_ROPE)
        if (kq == 0) {
#pragma unroll
            for (int j = 0; j < SH; ++j) {
                const int pg = slot[j] >= 0 ? slot[j] / a.page_size : 0, at = slot[j] - pg * a.page_size;
                cell_of[16 * j + r] = slot[j] >= 0 ? (((long long)pg * a.nkvh * a.page_size + at) << (a.half_log + 1)) : -1;
            }
        }
    auto put = [&](int at, const float* v) {
        uint16_t b[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) b[e] = __builtin_bit_cast(uint16_t, __float2bfloat16(v[e]));
        *reinterpret_cast<uint2*>(mine + r * ROW + at + 8 * kq) = uint2{(unsigned)b[0] | ((unsigned)b[1] << 16), (unsigned)b[2] | ((unsigned)b[3] << 16)};
    };
    // the rotation of 16 rows is fetched while the 16 before are stored
    v4f cs[ONT], sn[ONT];
    auto fetch_rotation = [&](int j) {
#pragma unroll
        for (int nt = 0; nt < ONT; ++nt) {
            const size_t at = ((size_t)pos[j] << a.half_log) + ((c0 + 16 * nt) & ((1 << a.half_log) - 1)) + 4 * kq;
            cs[nt] = *reinterpret_cast<const v4f*>(a.cos_t + at);
            sn[nt] = *reinterpret_cast<const v4f*>(a.sin_t + at);
        }
    };
    if constexpr (EPI == EPI_ROPE) fetch_rotation(0);
#pragma unroll
    for (int j = 0; j < SH; ++j) {
#pragma unroll
        for (int nt = 0; nt < ONT; ++nt) {
            float v[4], u[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = acc[nt][j][e];
                if constexpr (PAIRS) u[e] = acc[nt + ONT][j][e];
                if constexpr (EPI == EPI_SWIGLU) v[e] = silu_mul_fast(v[e], u[e]);
            }
            if constexpr (EPI == EPI_ROPE) {
                if (((c0 + 16 * nt) >> a.half_log) < a.nh + a.nkvh) {          // 16 pairs lie in one head
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float x = v[e], y = u[e];
                        v[e] = x * cs[nt][e] - y * sn[nt][e];
                        u[e] = x * sn[nt][e] + y * cs[nt][e];
                    }
                }
                put(32 * (nt + ONT), u);
            }
            put(32 * nt, v);
        }
        if constexpr (EPI == EPI_ROPE)
            if (j + 1 < SH) fetch_rotation(j + 1);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < (16 * PER_ROW + 63) / 64; ++i) {
            const int q = lane + 64 * i, lr = q / PER_ROW, ch = q - lr * PER_ROW;
            const int m = row0 + 16 * j + lr, n = c0 + 8 * (ch % (2 * ONT));
            if ((16 * PER_ROW % 64 != 0 && q >= 16 * PER_ROW) || m >= a.M || n >= NO) continue;
            const uint4 w = *reinterpret_cast<const uint4*>(mine + lr * ROW + 16 * ch);
            if constexpr (EPI == EPI_ROPE) {
                const int head = n >> a.half_log, col = (n & ((1 << a.half_log) - 1)) + (ch < 2 * ONT ? 0 : 1 << a.half_log);
                uint16_t* to = a.C + (size_t)m * a.ldc + ((size_t)head << (a.half_log + 1));
                if (head >= a.nh) {                                // (nothing reads a key or a value in C)
                    const bool v = head >= a.nh + a.nkvh;
                    const long long cell = cell_of[16 * j + lr];
                    if (cell < 0) continue;
                    to = (v ? a.vcache : a.kcache) + cell + (((long long)(head - a.nh - (v ? a.nkvh : 0)) * a.page_size) << (a.half_log + 1));
                }
                *reinterpret_cast<uint4*>(to + col) = w;
            } else {
                *reinterpret_cast<uint4*>(a.C + (size_t)m * a.ldc + n) = w;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <typename T, int EPI> int launch(TilesArgs a, hipStream_t stream) {
    a.tiles_m = (a.M + T::BM - 1) / T::BM;
    a.tiles_n = EPI != EPI_BF16 ? (a.N / 2 + T::BN / 2 - 1) / (T::BN / 2) : (a.N + T::BN - 1) / T::BN;
    const int groups = (a.tiles_m + 7) / 8;
    a.group_m = (a.tiles_m + groups - 1) / groups;
    const long long blocks = (long long)a.tiles_m * a.tiles_n;
    if (blocks > (1LL << 30)) return IC_ERR_ARG;
    if constexpr (T::takes(EPI)) {
        hipLaunchKernelGGL((gemm_tiles_kernel<T, EPI>), dim3((unsigned)blocks), dim3(T::WAVES * 64), 0, stream, a);
        return ic_launch_status();
    }
    return IC_ERR_ARG;
}

// The tiles, smallest first, and what one costs in microseconds: FIXED + rounds * (ROUND + stages * STAGE * (1 + FULL * x)), where x is the part of
// the compute units (256 of them where this was fitted) that have a block and a round is one block a unit (two of 64 x 32 and 64 x 64, which then share it: 1.7 times the stage).
// Fitted to 6,900 timed products (17 pairs of N in 512..32,768 and K in 512..16,384, 33..16,384 rows, weights out of memory); the tile with the least
// cost loses 0.7 % to the best one on average and 5 % at the 95th percentile.  64 x 32 is for few rows of narrow matrices, where only many small tiles
// reach all units (64 x 6,912 x 2,304: 15.0 us with 64 x 64, 11.8), 64 x 96 and 128 x 64 likewise (200 x 4,608 x 4,096: 25.4 -> 21.3).  Tried and not
// kept: 192 x 256, 96 x 192, 96 x 256, 64 x 192; two lines of 64 k a stage; more stages of the small tiles (no faster: what bounds them is the rate at
// which one unit takes bytes).
#define IC_TILES(X) \
    /* number, FIXED, STAGE, FULL, ROUND, tile: BM, BN, WM, WN, WK, STAGES */ \
    X(0, 2.76, 0.112, 0.65, 0.00, 64, 32, 2, 1, 2, 6) \
    X(1, 2.60, 0.198, 0.29, 0.00, 64, 64, 2, 1, 2, 4) \
    X(2, 2.07, 0.252, 0.20, 0.89, 64, 96, 2, 2, 1, 7) \
    X(3, 2.67, 0.256, 0.41, 0.43, 128, 64, 2, 2, 1, 6) \
    X(4, 2.51, 0.315, 0.21, 0.50, 64, 128, 2, 2, 1, 6) \
    X(5, 2.35, 0.332, 0.29, 1.04, 96, 128, 2, 2, 1, 5) \
    X(6, 2.69, 0.385, 0.34, 0.98, 128, 128, 2, 2, 1, 5) \
    X(7, 3.04, 0.467, 0.39, 0.89, 192, 128, 2, 2, 1, 3) \
    X(8, 3.43, 0.525, 0.28, 0.47, 128, 192, 2, 2, 1, 4) \
    X(9, 3.41, 0.574, 0.28, 0.96, 160, 192, 2, 2, 1, 3) \
    X(10, 2.90, 0.575, 0.35, 1.89, 256, 128, 2, 2, 1, 3) \
    X(11, 3.39, 0.662, 0.25, 0.83, 128, 256, 2, 2, 1, 3) \
    X(12, 3.69, 0.708, 0.29, 1.53, 160, 256, 2, 2, 1, 3) \
    X(13, 4.33, 0.956, 0.24, 0.00, 256, 192, 2, 2, 1, 2) \
    X(14, 6.27, 1.084, 0.30, 0.00, 256, 256, 2, 2, 1, 2)

constexpr int kTiles = 15;

struct TileCost { int bm, bn, blocks_per_unit; bool takes[3]; double fixed, stage, full, round; };
constexpr TileCost kCosts[kTiles] = {
#define X(I, FIXED, STAGE, FULL, ROUND, ...) {Tile<__VA_ARGS__>::BM, Tile<__VA_ARGS__>::BN, Tile<__VA_ARGS__>::BLOCKS_PER_CU, {true, Tile<__VA_ARGS__>::takes(EPI_SWIGLU), Tile<__VA_ARGS__>::takes(EPI_ROPE)}, FIXED, STAGE, FULL, ROUND},
    IC_TILES(X)
#undef X
};

// units: compute units of the device or partition; memory serves each its share of the whole chip's rate.
double cost_of(const TileCost& t, int M, int N, int K, int mode, int units) {
    const long long tm = (M + t.bm - 1) / t.bm, tn = mode != EPI_BF16 ? (N / 2 + t.bn / 2 - 1) / (t.bn / 2) : (N + t.bn - 1) / t.bn;
    const double tiles = (double)(tm * tn), x = tiles / units, stages = K / 64;
    double rounds = 1.0, busy = x < 1.0 ? x : 1.0, shared = 1.0, again = 0.0;
    if (x > 1.0) {
        rounds = __builtin_ceil(x / t.blocks_per_unit);
        // tiles that share a unit have no ROUND of their own, but every further round launches, fetches and stores before and after its stages: 2.3 us
        // (64 x 64 tiles with K = 64: 4.6 us in one round, 7.3 in two, 10.5 in three, 14.2 in five).  Without it short walks ran in many rounds of them.
        if (t.blocks_per_unit > 1) { shared = 1.7; again = 2.3 * (rounds - 1.0); }
    }
    const double walk = t.fixed + rounds * (t.round + stages * t.stage * (1.0 + t.full * busy) * shared) + again;
    // the weights come from memory once, and about half of them again for every further row tile (blocks of one column of tiles seldom run abreast);
    // narrow tiles of pairs read them in pieces of 32 rows and less, which memory serves more slowly (64 x 32,768 x 4,096: 83 us against 63)
    const double read = 3.0 + 2.0 * N * K * (1.0 + 0.5 * (tm < 4 ? tm - 1 : 3)) * (mode != EPI_BF16 && t.bn <= 64 ? 1.35 : 1.0) / (7e6 * units / 256.0);
    return walk > read ? walk : read;
}

int best_tile(int M, int N, int K, int mode, int units, double* cost) {
    int best = 0;
    for (int i = 0; i < kTiles; ++i) {
        if (!kCosts[i].takes[mode]) continue;
        const double c = cost_of(kCosts[i], M, N, K, mode, units);
        if (i == 0 || c < *cost) { *cost = c; best = i; }
    }
    return best;
}

template <int EPI> int by_number(int tile, const TilesArgs& a, hipStream_t stream) {
    switch (tile) {
#define X(I, FIXED, STAGE, FULL, ROUND, ...) case I: return launch<Tile<__VA_ARGS__>, EPI>(a, stream);
        IC_TILES(X)
#undef X
    }
    return IC_ERR_ARG;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Whole stages of K, 16-byte pieces of every row, byte offsets within 32 bits.  cols: columns of C.
bool takes(int M, int N, int K, int lda, int ldw, int cols, int ldc, int mode) {
    if (M <= 0 || M > (1 << 30) || N <= 0 || N > (1 << 30) || K <= 0 || K % 64 || lda < K || ldw < K || lda % 8 || ldw % 8) return false;
    if (N % (mode != EPI_BF16 ? 16 : 8) || ldc < cols || ldc % 8) return false;
    if ((long long)lda * 2 * 256 >= (1LL << 31) || (long long)ldw * 2 * (mode != EPI_BF16 ? N : 256) >= (1LL << 32)) return false;
    return (long long)((M + 63) / 64) * ((N + 63) / 64) < (1LL << 28);
}

int run(const TilesArgs& a, int mode, int tile, hipStream_t stream) {
    if (mode == EPI_ROPE) return by_number<EPI_ROPE>(tile, a, stream);
    return mode == EPI_SWIGLU ? by_number<EPI_SWIGLU>(tile, a, stream) : by_number<EPI_BF16>(tile, a, stream);
}

TilesArgs plain_args(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc) {
    return TilesArgs{(const uint16_t*)A, (const uint16_t*)W, (uint16_t*)C, M, N, K, lda, ldw, ldc};
}

int rope_run(const void* A, const void* W, void* C, int M, int K, int lda, int ldw, int ldc, const int* positions, const int* slots, const float* cos_t,
             const float* sin_t, void* kcache, void* vcache, int nh, int nkvh, int dh, int page_size, int tile, hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!positions || !slots || tile >= kTiles ||
        !ic_gemm_tiles_rope_supported(A, W, C, M, K, lda, ldw, ldc, cos_t, sin_t, kcache, vcache, nh, nkvh, dh, page_size)) return IC_ERR_ARG;
    const int N = (nh + 2 * nkvh) * dh;
    TilesArgs a = plain_args(A, W, C, M, N, K, lda, ldw, ldc);
    a.positions = positions, a.slots = slots, a.cos_t = cos_t, a.sin_t = sin_t;
    a.kcache = (uint16_t*)kcache, a.vcache = (uint16_t*)vcache;
    a.nh = nh, a.nkvh = nkvh, a.page_size = page_size;
    while ((2 << a.half_log) < dh) ++a.half_log;
    double cost = 0.0;
    return run(a, EPI_ROPE, tile >= 0 ? tile : best_tile(M, N, K, EPI_ROPE, compute_units(), &cost), stream);
}

}  // namespace

IC_EXPORT int ic_gemm_tiles_supported(int M, int N, int K, int lda, int ldw, int ldc, int mode) {
    return (mode == EPI_BF16 || mode == EPI_SWIGLU) && takes(M, N, K, lda, ldw, mode == EPI_SWIGLU ? N / 2 : N, ldc, mode);
}

// Heads of 32, 64, 128, .. entries, so that 16 neighbouring pairs lie in one head and a pair's head is a shift away.
IC_EXPORT int ic_gemm_tiles_rope_supported(const void* A, const void* W, const void* C, int M, int K, int lda, int ldw, int ldc, const float* cos_t,
                                           const float* sin_t, const void* kcache, const void* vcache, int nh, int nkvh, int dh, int page_size) {
    if (nh <= 0 || nkvh <= 0 || dh < 32 || dh > 1024 || (dh & (dh - 1)) || page_size <= 0 || (long long)(nh + 2LL * nkvh) * dh >= (1LL << 30)) return 0;
    const void* const all[7] = {A, W, C, cos_t, sin_t, kcache, vcache};
    for (const void* p : all)
        if (!p || !aligned16(p)) return 0;
    return takes(M, (nh + 2 * nkvh) * dh, K, lda, ldw, nh * dh, ldc, EPI_ROPE);
}

// Whether the own kernel is the faster one: its cost against what the library's product (and the kernel that follows it, where the epilogue has that) would
// take.  The library's times jump between neighbouring sizes, so the lines are fitted to 3,900 timed products with weights out of memory (150 pairs of N in
// 64..32,768 and K in 64..16,384, 33..16,384 rows; the library's first choice of algorithm).  What they choose loses 1.4 % to the faster of the two on
// average and is over 3 % slower than the library in 3.7 % of the products, over 10 % in 0.8 % (the own kernel everywhere: 3.3 % lost, the library everywhere:
// 39 %):
//   up to 64 rows the library splits K over the chip where K is a multiple of 256: about 11 us, the weights and the products at the rates below, however
//   long K is, while the own kernel's walk grows with K.  64 x 4,096 x 14,336: 40 us against 52, 48 x 2,048 x 11,264: 20 against 36; on this side of
//   the line 64 x 2,304 x 2,304: 9.9 -> 7.4.  Other K it does not split, or badly (33 x 2,304 x 5,760: 25.4 -> 17.4);
//   there, and up to 512 rows, where its times jump most (4,096 x 16,384: 50 us for 65 rows, 69 for 96, 93 for 160, 65 for 256; own 42, 45, 67, 72), only walks far
//   beyond a split over the whole chip go to it (256 x 256 x 16,384: 17 against 30; on this side 256 x 1,536 x 3,840: 14.4 -> 10.3);
//   more rows: where its 256 x 256 tiles, which spend some 6 % less on a stage than the own ones, fit about as well as the own best tile: whole tiles of
//   columns, K of 1,024 and more (shorter walks are mostly the way out), no ragged last round behind more than four (16,384 x 4,608 x 4,096: 556 -> 452)
//   (8,192 x 4,096 x 14,336: 615 us against 704; 2,048 x 6,912 x 2,304: 51 against 58; else 1,045 x 2,560 x 1,536: 16.9 -> 12.1, 2,048 x 2,304 x 2,304: 28.0 -> 23.1);
//   a single stage of K in more than one round, where nothing is left to overlap with a tile's way out (3,300 x 4,096 x 64: 10.9 against 15.2; in one round
//   the own kernel is ahead, 1,300 x 2,304 x 64: 5.7 -> 4.9).
// The gated unit in the epilogue saves its kernel, 3 us and more, and pays from 33 rows on but for long K as above (48 x 2,048 x 12,288: 24 us against 39) and for
// 190 MB of weights and more in rows of 12 KB and more, which few row tiles read more slowly than the library (96 x 16,384 x 6,144: 54 against 67; else
// 1,045 x 7,680 x 1,536: 42.8 -> 28.0; 2,048 x 11,520 x 2,304: 130 -> 98; 16,384 x 32,768 x 4,096: 3,195 -> 3,007).  So does rotary and cache write behind QKV
// (64 rows of the 2B shape 18.3 -> 12.5, 1,045 rows of the 1B shape 21.5 -> 15.5, 2,048 of the 8B shape 78.6 -> 69.6), but for sizes that the largest tile
// fits best, which this epilogue does not have.
IC_EXPORT int ic_gemm_tiles_pays_on(int M, int N, int K, int mode, int units) {
    if (M <= 32 || M > (1 << 30) || N <= 0 || N > (1 << 30) || K <= 0 || units <= 0 || mode < EPI_BF16 || mode > EPI_ROPE) return 0;
    const double t = (double)((M + 255) / 256) * ((N + 255) / 256), fill = t / (units * __builtin_ceil(t / units)), part = units / 256.0;
    if (mode != EPI_BF16 && K > 8192 && fill >= 0.93) return 0;
    double cost = 0.0;
    if (mode == EPI_ROPE) return kCosts[best_tile(M, N, K, EPI_SWIGLU, units, &cost)].takes[EPI_ROPE];
    const TileCost& own = kCosts[best_tile(M, N, K, mode, units, &cost)];
    const double weights = 2.0 * N * K / part, products = weights * M;     // bytes, operations for the whole chip's rates below
    if (M <= 64 && K % 256 == 0) {
        const double read = weights / 7.2e6, unit = mode == EPI_SWIGLU ? 3.0 + 0.75e-6 * M * N : 0.0;
        if ((cost > read ? cost : read) > 11.35 + weights / 9.06e6 + products / 5.0e9 + unit) return 0;
    }
    if (mode == EPI_SWIGLU) return !(M <= 96 && K >= 6144 && K % 256 == 0 && 2.0 * N * K >= 1.9e8);
    if (K == 64 && (double)((M + own.bm - 1) / own.bm) * ((N + own.bn - 1) / own.bn) > (double)units * own.blocks_per_unit) return 0;
    const double over = 6.0 + (products / 0.6e9 > weights / 4e6 ? products / 0.6e9 : weights / 4e6);
    if (M <= 512) return cost <= 1.6 * over;
    const bool whole = N % 256 == 0 && K >= 1024 && !(t > 4.0 * units && fill < 0.92);
    return cost <= 2.0 * over && !(whole && cost > 0.94 * cost_of(kCosts[kTiles - 1], M, N, K, EPI_BF16, units));
}

IC_EXPORT int ic_gemm_tiles_pays(int M, int N, int K, int mode) { return ic_gemm_tiles_pays_on(M, N, K, mode, compute_units()); }

IC_EXPORT int ic_gemm_tiles_plan_on(int M, int N, int K, int mode, int units) {
    double cost = 0.0;
    return M > 0 && N > 0 && K > 0 && units > 0 && mode >= EPI_BF16 && mode <= EPI_ROPE ? best_tile(M, N, K, mode, units, &cost) : -1;
}

IC_EXPORT int ic_gemm_tiles_plan(int M, int N, int K, int mode) { return ic_gemm_tiles_plan_on(M, N, K, mode, compute_units()); }

IC_EXPORT int ic_gemm_tiles(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, int mode, hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!A || !W || !C || !ic_gemm_tiles_supported(M, N, K, lda, ldw, ldc, mode) || !aligned16(A) || !aligned16(W) || !aligned16(C)) return IC_ERR_ARG;
    double cost = 0.0;
    return run(plain_args(A, W, C, M, N, K, lda, ldw, ldc), mode, best_tile(M, N, K, mode, compute_units(), &cost), stream);
}

IC_EXPORT int ic_gemm_tiles_cfg(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc, int mode, int tile,
                                hipStream_t stream) {
    if (M <= 0) return IC_OK;
    if (!A || !W || !C || tile < 0 || tile >= kTiles || !ic_gemm_tiles_supported(M, N, K, lda, ldw, ldc, mode) || !aligned16(A) || !aligned16(W) ||
        !aligned16(C)) return IC_ERR_ARG;
    return run(plain_args(A, W, C, M, N, K, lda, ldw, ldc), mode, tile, stream);
}

IC_EXPORT int ic_gemm_tiles_rope(const void* A, const void* W, void* C, int M, int K, int lda, int ldw, int ldc, const int* positions, const int* slots,
                                 const float* cos_t, const float* sin_t, void* kcache, void* vcache, int nh, int nkvh, int dh, int page_size,
                                 hipStream_t stream) {
    return rope_run(A, W, C, M, K, lda, ldw, ldc, positions, slots, cos_t, sin_t, kcache, vcache, nh, nkvh, dh, page_size, -1, stream);
}

IC_EXPORT int ic_gemm_tiles_rope_cfg(const void* A, const void* W, void* C, int M, int K, int lda, int ldw, int ldc, const int* positions, const int* slots,
                                     const float* cos_t, const float* sin_t, void* kcache, void* vcache, int nh, int nkvh, int dh, int page_size, int tile,
                                     hipStream_t stream) {
    if (tile < 0) return IC_ERR_ARG;
    return rope_run(A, W, C, M, K, lda, ldw, ldc, positions, slots, cos_t, sin_t, kcache, vcache, nh, nkvh, dh, page_size, tile, stream);
}

// The product by the kernel that is faster for it, as timed (ic_product_tune) or by the rule: this file's or the library's, in float32 gemm_f32.hip's or the library's.
IC_EXPORT int ic_product(const void* A, int a_dtype, const void* W, void* C, int c_dtype, int M, int N, int K, int lda, int ldw, int ldc, float alpha,
                         void* workspace, long long workspace_bytes, hipStream_t stream) {
    if (a_dtype == IC_BF16 && c_dtype == IC_BF16 && alpha == 1.0f && A && W && C && ic_gemm_tiles_supported(M, N, K, lda, ldw, ldc, EPI_BF16) &&
        aligned16(A) && aligned16(W) && aligned16(C)) {
        const int timed = ic_product_timed(M, N, K, lda, ldw, ldc);
        if (timed >= 0 ? timed : ic_gemm_tiles_pays(M, N, K, EPI_BF16)) return ic_gemm_tiles(A, W, C, M, N, K, lda, ldw, ldc, EPI_BF16, stream);
    }
    if (a_dtype == IC_F32 && c_dtype == IC_F32)
        return ic_product_f32(A, W, C, M, N, K, lda, ldw, ldc, alpha, workspace, workspace_bytes, workspace, workspace_bytes, stream);
    return ic_matmul(A, a_dtype, W, C, c_dtype, M, N, K, lda, ldw, ldc, alpha, workspace, workspace_bytes, stream);
}
