// All layers of a decode step in one launch, for up to 8 rows in bfloat16 (sizes: `instance` below, rows: `most_rows`).
//
// Why: with few rows a layer is five or six kernels of 5..12 us each, of which 2..5 go by before the first weights are there and after the last block has ended; the
// 1B shape's layer brings 48 MB, 6.8 us at 7.1 TB/s, and took 28.  Here one block a compute unit stays for the whole step.  Its 12 waves have two trades:
//   8 stream.  They send a task's weights (keys, values) into registers before the rows that they multiply are there, take one step on the matrix cores when
//     they are (operands as in gemm_rows.hip), and leave their halves of the results in LDS.
//   4 control.  They fetch the rows from where other blocks write them into LDS, sum the streaming waves' results, and write the block's share.  Loads return in
//     order to a wave, so what waits for other blocks must not stand behind weights: hence waves of their own.
// Phases of a layer: QKV with rotary and cache write; attention; if heads are walked in pieces, the pieces together; O into the residual stream; gate/up with the unit;
// down into the residual stream.  The norms are split over the products around them as in the few-row kernels (x times the weight and sums of squares on one side, row
// factors on the other).
//
// Handing on.  Every value that a block hands on has a place of its own per layer and step, which is all ones ("empty") when the step starts (chain_start_kernel) and is written
// once, past the caches of the die (agent scope).  Who needs rows reads them past the caches again and again until nothing in them is empty: one way to memory and back, where
// counters cost a wait for the writes, an atomic, a question and then the read (1B shape, one row: 28.4 -> 23.6 us a layer).  What is sent ahead waits until a block's
// results are written (a second meeting of the waves): with loads in front of them results come late (1,060 -> 1,280 us a step of the 1B shape).
//
// Who takes part.  A block waits only for blocks that run: those that have come join at the start, and after a while nobody else does (other work fills the device, or
// another such kernel does); tasks are dealt to those n, what they compute does not depend on n.  The while: what the missing ones cost, which is a step's time for every
// round beyond the first in which n blocks do the tasks of G, so that such a step takes about twice its best at most; a millisecond at least.  (Closing after a millisecond whatever n is, with
// the layers in launches of 4, 13 and 26, steps beside another engine's decoding: the slowest of 150 took 13.9, 37 and 72 ms, and 3.6, 4.8 and 6.1 so; of whole steps the
// slowest is 3.3 either way.)
// Beside other streams' work (1B shape, one row of 258 keys; kernel by kernel / so, us a step): another engine's prompts of 2,048 (2B shape) 3,700 / 1,200, its steps of 7 rows 2,450 /
// 2,950, products of 4,096^3 13,800 / 1,450, of 16,384^3 706,000 / 18,000; two engines of 4, 12 and 24 layers 426 / 294, 923 / 750, 1,680 / 1,430.  The blocks fill the units'
// registers, so other work runs between steps: those prompts take 181 ms instead of 15 meanwhile, the products of 4,096^3 360 us each instead of 110.  In launches
// of 20 layers 97 ms and 250 us, for 0.3 % of a step alone and 1.1..1.8 times a step beside others; left so.
//
// One row, us a step, kernel by kernel / so: 1B shape at 100, 600, 2,000 keys 1,380 / 995, 1,535 / 1,142, 1,553 / 1,229; 2B shape 1,621 / 1,333, 1,722 / 1,453,
// 1,839 / 1,507.  Four rows: 1,514 / 1,162, 1,628 / 1,344, 1,725 / 1,423; 1,632 / 1,446, 1,730 / 1,567, 2,027 / 1,859.  What bounds it: each phase is about 1 us of products and
// results and 1.5..2.5 for the slowest block's results to be seen, in which memory idles or brings the next weights; rows are read by every block, so it grows with them
// (`most_rows`).
// Tried and no faster: two questions under way at a time (1,062 -> 1,124 us), pauses between them (1,080 at 4 x 64 cycles), up to 8 copies of what all blocks read
// (1,063, 16: 1,097), loads for the next phase before a block's results are written (2B shape 1,458 -> 1,465), gate/up's first lines already while attention ends (1,448: what
// it saves there the merging of the pieces loses), keys and values with QKV's weights (1,522).
#include "decode_chain.h"
#include "infinicore_infer_variants.h"
#include "attn_decode_blocks.h"
#include <algorithm>
#include <type_traits>

namespace {

typedef __bf16 ch_v8b __attribute__((ext_vector_type(8)));
typedef float ch_v4f __attribute__((ext_vector_type(4)));
typedef const void __attribute__((address_space(1)))* ch_gptr;
typedef void __attribute__((address_space(3)))* ch_lptr;
typedef unsigned long long ch_u64;

constexpr int kStream = 8;                 // waves that bring weights, keys and values
constexpr int kControl = 4;                // waves that wait for other blocks, stage rows and write results
constexpr int kThreads = 64 * (kStream + kControl);
constexpr int kRing = 24;                  // 16-byte registers of a streaming lane: 192 KB of a unit in flight at most (28: no faster; 30 do not fit)
constexpr int kLinesAhead = 12;            // lines of a product that are sent ahead at most
constexpr int kCounters = 32;              // of the blocks that have come, a cache line each
constexpr int kLineWords = 32;
constexpr unsigned kClosed = 0x10000u;
constexpr int kMaxPieces = 40;              // of a block's attention work
constexpr int DH = 64;                     // elements of a head
constexpr int kMaxGroup = 4;               // query heads of a kv head
constexpr int kMaxPageIds = 2048;
constexpr int kUnit = 64;                  // keys of a unit of attention work
constexpr int kGaveUp = 2 * kCounters * kLineWords;     // not 0: a block has given up a wait
constexpr int kSyncWords = kGaveUp + kLineWords;
constexpr unsigned kJoinTicks = 100000;                 // 1 ms of the 100 MHz clock
constexpr unsigned kLayerTicks = 2500;                  // a layer with a block on every unit, about
constexpr int kFarLoad = 16;                // sc1: past this die's caches
constexpr int kPace = 10;                   // loads of a streaming wave in flight while it sends ahead (3: 1,532 us a step of the 2B shape, 6: 1,489, 10: 1,460, 16: 1,458)
// A wait ends when blocks that run have written.  Should it not end after some seconds (kChainTries questions) all the same, the block gives up: its results, with them the
// step's logits, are NaN, no keys and values are cached of what came from it, and the caller is told (gave_up).

struct Layout {                            // byte offsets within one entry's scratch
    long long y_in, ss_in, q, kv, attn, acc, ml, y_mid, ss_mid, act, stride;
};

struct ChainArgs {
    const ChainEntry* entries;
    int n_entries, T, d, nh, nkv, di, page_size, ow;
    PageDivider div;
    float scale, rscale, eps_in, eps_mid;
    const int *positions, *slots, *token_req, *tables;
    int bt_stride;
    const float *cos_t, *sin_t;
    float* x;
    unsigned char* scratch;
    Layout at;
    unsigned* sync;
    int* gave_up;
    int tries;
    bf16* y_out;
    float* ss_out;
    int G, cols, t_qkv, t_res, t_gu;
    int rows_bytes, red_floats;
};

// The kernel's arguments and the layers' table where they lie, read by scalar loads at each use: held in registers over the loop they would not fit.
typedef const ChainArgs __attribute__((address_space(4)))* Args;
__device__ __forceinline__ Args again(Args a) { asm volatile("" : "+s"(a)); return a; }
__device__ __forceinline__ int page_of(Args a, int key) {
    const unsigned mul = a->div.mul;
    return (int)((unsigned)(((unsigned long long)(unsigned)key * mul + mul) >> 32) >> a->div.shift);
}

__device__ __forceinline__ ch_v8b ch_op(const uint4& v) { return __builtin_bit_cast(ch_v8b, v); }
template <typename V> __device__ __forceinline__ void st_far(V* p, V v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <typename V> __device__ __forceinline__ V ld_far(const V* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// What blocks hand on is written once into memory that is all ones at the start of the step ("empty"), and never all ones: a NaN of that pattern becomes another.
__device__ __forceinline__ uint16_t full_bits(float v) { const uint16_t b = f32_to_bf16_bits(v); return b == 0xffffu ? (uint16_t)0x7fc0u : b; }
__device__ __forceinline__ void put(bf16* p, float v) { st_far((unsigned short*)p, full_bits(v)); }
__device__ __forceinline__ float full_word(float v) { return __float_as_uint(v) == ~0u ? __uint_as_float(0x7fc00000u) : v; }
__device__ __forceinline__ void put(float* p, float v) { st_far((unsigned*)p, __float_as_uint(full_word(v))); }
// Not zero: one of the two halves is empty.
__device__ __forceinline__ unsigned empty_halves(unsigned v) { const unsigned z = ~v; return (z - 0x00010001u) & v & 0x80008000u; }
// LDS written before is seen by the other waves after; loads from memory stay in flight.
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The same value, which the compiler takes for another: what is computed from it stays inside the loop over the layers, where registers are scarce.
__device__ __forceinline__ int again_v(int v) { asm volatile("" : "+v"(v)); return v; }
__device__ __forceinline__ int again_s(int v) { asm volatile("" : "+s"(v)); return v; }

struct Piece { int row, kvh, lo, hi, slot, page_lo, page_off, pos; };

// What a block knows about the step, in LDS.
struct Shared {
    int n, rank;                           // blocks that take part, this one's number
    int tries;                             // questions of a wait; -1: one was given up, no other lasts
    int n_pieces, n_ids;
    int direct, workers;                   // 1: a block walks whole heads; blocks that walk
    int tiles[kChainMaxRows], before[kChainMaxRows + 1];      // units of attention work: of a row's head, of the rows before
    float factor[kChainMaxRows];
    Piece piece[kMaxPieces];
    float own[kMaxPieces][kMaxGroup];      // scores of the step's own keys, units of log 2
    int ids[kMaxPageIds];
};
static_assert(sizeof(Shared) % alignof(ChainEntry) == 0, "the layers' table lies behind it");

// ---- streaming waves: products --------------------------------------------------------------------------------------------
// The four products of a layer.  RG: groups of 8 weight rows of a task; EPI as in gemm_rows.hip.
enum { QKV, OUT_PROJ, GATE_UP, DOWN };
// A pointer of the layers' table, which the block keeps in LDS (a scalar load of it misses once a layer).  To device memory, which the compiler cannot know:
// a load whose address may lie in LDS would also be waited for by who waits for LDS.
typedef const unsigned char __attribute__((address_space(1)))* Far;
__device__ __forceinline__ Far uniform(const void* p) {
    const ch_u64 v = (ch_u64)p;
    return (Far)((ch_u64)(unsigned)__builtin_amdgcn_readfirstlane((int)v) | (ch_u64)(unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32);
}
__device__ __forceinline__ uint4 stream16(Far p) {
    typedef unsigned ch_v4u __attribute__((ext_vector_type(4)));
    const ch_v4u v = __builtin_nontemporal_load((const ch_v4u __attribute__((address_space(1)))*)p);
    return uint4{v[0], v[1], v[2], v[3]};
}
template <int KIND> __device__ __forceinline__ int tasks_of(Args a) { return KIND == QKV ? a->t_qkv : KIND == GATE_UP ? a->t_gu : a->t_res; }
template <int KIND> __device__ __forceinline__ int depth_of(Args a) { return KIND == DOWN ? a->di : KIND == OUT_PROJ ? a->ow : a->d; }
template <int KIND> __device__ __forceinline__ Far weights_of(const ChainEntry* E) {
    return uniform(KIND == QKV ? E->w_qkv : KIND == OUT_PROJ ? E->w_o : KIND == GATE_UP ? E->w_gate_up : E->w_down);
}

// Byte offsets of this lane's rows of task t.
template <int KIND, int RG>
__device__ __forceinline__ void row_offsets(Args a, int t, int K, int lane, unsigned (&off)[RG]) {
    const int r8 = lane & 7, hi = (lane >> 3) & 1, kq = lane >> 4, col8 = 8 * (kq + 4 * hi);
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        int row, last;
        if constexpr (KIND == GATE_UP) {
            const int up = (g / (RG / 2)) * a->di;
            row = t * (4 * RG) + 8 * (g % (RG / 2)) + r8 + up;
            last = a->di - 1 + up;
        } else if constexpr (KIND == QKV) {
            const int pair = t * (RG / 2) + (g >> 1), per_head = DH >> 4;
            const int head = pair / per_head, j = 8 * (pair - head * per_head);
            row = head * DH + r8 + (head < a->nh + a->nkv ? j + (g & 1) * (DH >> 1) : 2 * j + 8 * (g & 1));
            last = (a->nh + 2 * a->nkv) * DH - 1;
        } else {
            row = t * a->cols + 8 * g + r8;
            last = min((t + 1) * a->cols, a->d) - 1;
        }
        off[g] = (unsigned)(row < last ? row : last) * (unsigned)(2 * K) + 2u * col8;
    }
}

// (What a slot holds that is not used is defined: with undefined registers in the branches the allocation goes astray.)
__device__ __forceinline__ void clear(uint4* slots, int n) {
#pragma unroll
    for (int i = 0; i < n; ++i) slots[i] = uint4{0, 0, 0, 0};
}

// More loads than these would stand in the way of what the control waves read and write.
template <int N> __device__ __forceinline__ void pace() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

template <int RG, int PACE = 63>
__device__ __forceinline__ void send_line(Far w, int line, const unsigned (&off)[RG], uint4* dst) {
    const Far b = w + 128 * line;
#pragma unroll
    for (int g = 0; g < RG; ++g) {
        dst[g] = stream16(b + off[g]);
        if constexpr (PACE < 63) pace<PACE>();
    }
    __builtin_amdgcn_sched_barrier(0);
}


template <int RG> constexpr int kLines = kRing / RG < kLinesAhead ? kRing / RG : kLinesAhead;      // of a product that the ring holds

// A task's first lines into the ring.
template <int KIND, int RG>
__device__ __forceinline__ void send_ahead(Args a, const ChainEntry* E, int t, int lane, int wave, uint4* ring) {
    a = again(a);
    lane = again_v(lane);
    wave = again_s(wave);
    const int K = depth_of<KIND>(a), nl = ((K >> 6) - wave + kStream - 1) / kStream;
    const Far w = weights_of<KIND>(E);
    unsigned off[RG];
    row_offsets<KIND, RG>(a, t, K, lane, off);
#pragma unroll
    for (int s = 0; s < kLines<RG>; ++s)
        if (s < nl) {
            send_line<RG, kPace>(w, wave + kStream * s, off, ring + s * RG);
        } else clear(ring + s * RG, RG);
}

template <int KIND, int RG>
__device__ __forceinline__ void multiply(Args a, const ChainEntry* E, int t, int lane, int wave, uint4* ring, const unsigned char* rows, float* red) {
    constexpr int S = kLines<RG>, OUT = RG * 64;
    a = again(a);
    lane = again_v(lane);
    wave = again_s(wave);
    const int r8 = lane & 7, hi = (lane >> 3) & 1, kq = lane >> 4;
    const int K = depth_of<KIND>(a), T = a->T;
    int left = ((K >> 6) - wave + kStream - 1) / kStream, l = wave;
    const unsigned char* const ap = rows + 128 * min(r8, T - 1) + 16 * (kq + 4 * hi);
    const int line_bytes = 128 * T;
    ch_v4f acc[RG];
#pragma unroll
    for (int g = 0; g < RG; ++g) acc[g] = ch_v4f{0.f, 0.f, 0.f, 0.f};
    auto use = [&](int s, int line) {
        const uint4 tok = *reinterpret_cast<const uint4*>(ap + line * line_bytes);
#pragma unroll
        for (int g = 0; g < RG; ++g) acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ch_op(ring[s * RG + g]), ch_op(tok), acc[g], 0, 0, 0);
    };
    if (left > S) {
        const Far w = weights_of<KIND>(E);
        unsigned off[RG];
        row_offsets<KIND, RG>(a, t, K, lane, off);
        while (left >= 2 * S) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                use(s, l + kStream * s);
                send_line<RG>(w, l + kStream * (s + S), off, ring + s * RG);
            }
            left -= S;
            l += kStream * S;
        }
        if (left > S) {
            const int more = left - S;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                use(s, l + kStream * s);
                if (s < more) send_line<RG>(w, l + kStream * (s + S), off, ring + s * RG);
            }
            left -= S;
            l += kStream * S;
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (s < left) use(s, l + kStream * s);
    if (hi == (kq >> 1)) {
#pragma unroll
        for (int g = 0; g < RG; ++g) *reinterpret_cast<ch_v4f*>(red + (2 * wave + hi) * OUT + g * 64 + 8 * r8 + 4 * (kq & 1)) = acc[g];
    }
}

// ---- attention work: who walks what --------------------------------------------------------------------------------------------
// Blocks walk whole heads (of one row and kv head) where that makes the longest walk at most this much longer than equal runs, which need a phase more to bring
// the pieces together.  Else the units (64 keys of a head) of all heads in a line are dealt to the workers in equal runs of one unit at least; a run that ends
// within a head leaves a piece of it, whose partial result has the place head + worker (no two pieces the same: from one to the next one of the two grows).
__host__ __device__ __forceinline__ bool walks_whole_heads(int heads, int G, int longest, int units) { return (heads + G - 1) / G * longest - units / G <= 5; }
__host__ __device__ __forceinline__ int workers_of(bool whole, int heads, int units, int G) { return whole ? (heads < G ? heads : G) : units < G ? units : G; }
__host__ __device__ __forceinline__ int units_of(int position) { return (position + kUnit) / kUnit; }      // of a head whose last key is there
__host__ __device__ __forceinline__ int first_unit(int w, int units, int workers) { return (int)((long long)w * units / workers); }
__host__ __device__ __forceinline__ int worker_of(int u, int units, int workers) { return (int)((unsigned)((u + 1) * workers - 1) / (unsigned)units); }

// Of one worker at most, over all steps of so many heads and at most so many units.
__host__ __device__ __forceinline__ long long most_pieces(long long heads, long long units, int G) {
    const long long run = (units + G - 1) / G + 1, whole = (heads + G - 1) / G;
    return whole > run ? whole : run < heads ? run : heads;
}

// add(row, kv head, first key, key after the last, place) for every piece of worker w; before[r]: units of the rows before r.
template <typename Add>
__host__ __device__ __forceinline__ void for_pieces(int w, bool whole, int workers, int rows, int nkv, const int* positions, const int* tiles, const int* before, Add add) {
    if (w >= workers) return;
    if (whole) {
        for (int s = w; s < rows * nkv; s += workers) { const int row = s / nkv; add(row, s - row * nkv, 0, positions[row] + 1, s); }
        return;
    }
    const int end = first_unit(w + 1, before[rows], workers);
    int row = 0;
    for (int u = first_unit(w, before[rows], workers); u < end;) {
        while (u >= before[row + 1]) ++row;
        const int in = u - before[row], kvh = in / tiles[row], tile = in - kvh * tiles[row];
        const int take = tiles[row] - tile < end - u ? tiles[row] - tile : end - u, hi = (tile + take) * kUnit;
        add(row, kvh, tile * kUnit, hi < positions[row] + 1 ? hi : positions[row] + 1, row * nkv + kvh + w);
        u += take;
    }
}

// By one thread: worker w's pieces.
__device__ void plan_pieces(Args a, Shared& sh, int w) {
    int np = 0, ids = 0;
    for_pieces(w, sh.direct, sh.workers, a->T, a->nkv, a->positions, sh.tiles, sh.before, [&](int row, int kvh, int lo, int hi, int slot) {
        Piece& p = sh.piece[np++];
        p.row = row; p.kvh = kvh; p.lo = lo; p.hi = hi; p.slot = slot;
        p.pos = a->positions[row];
        p.page_lo = page_of(a, lo);
        p.page_off = ids;
        ids += page_of(a, hi - 1) - p.page_lo + 1;
    });
    sh.n_pieces = np;
    sh.n_ids = ids;
}

template <int GQ> struct Heads {
    static constexpr int LPK = DH / 8;                       // lanes that share a key's row
    static_assert((GQ + 2) * LPK <= 64, "a piece's queries, its new key and value are one chunk");
    // One query head a kv head: a lane group of LPK walks every KPW-th key.  Several: tiles of 32 keys on the matrix cores.
    static constexpr bool TILES = GQ > 1;
    static constexpr int KPW = 64 / LPK, KPB = KPW * kStream;
    static constexpr int U = 2;                              // keys of a lane group in a stage
    static constexpr int NV = 32 * LPK / 64;                 // loads of a tile of keys
    static constexpr int SLOTS = TILES ? 2 * NV : 2 * U;     // of the ring, for a stage
    static constexpr int STEP = TILES ? 32 * kStream : U * KPB;              // keys of a stage of all waves
    static constexpr int S = TILES ? kRing / SLOTS : 6;         // stages in flight
    static constexpr int STATE = GQ * (DH + 2);
    static constexpr int VS = DH + 8;                        // row stride of a tile in LDS
    static constexpr int TILE_BYTES = TILES ? kStream * 32 * VS * 2 : 0;
};

__device__ __forceinline__ Piece piece_of(const Shared& sh, int i) {
    const Piece p = sh.piece[i];
    auto one = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    return Piece{one(p.row), one(p.kvh), one(p.lo), one(p.hi), one(p.slot), one(p.page_lo), one(p.page_off), one(p.pos)};
}

// Stage `stage` of a piece's cached keys and values; keys beyond them read the last one.
template <int GQ>
__device__ __forceinline__ void send_keys(Args a, const Shared& sh, const Piece& p, Far kc, Far vc, int stage, int lane, int wave, uint4* dst) {
    using H = Heads<GQ>;
    a = again(a);
    lane = again_v(lane);
    const int sub = lane % H::LPK, grp = lane / H::LPK;
    const int hi = min(p.hi, p.pos);
    const int ps = a->page_size;
    const unsigned head_bytes = (unsigned)ps * (2 * DH), page_bytes = (unsigned)a->nkv * head_bytes;
    kc += (size_t)p.kvh * head_bytes;
    vc += (size_t)p.kvh * head_bytes;
    constexpr int N = H::SLOTS / 2;
    const int first = p.lo + stage * H::STEP + (H::TILES ? 32 * wave : H::KPW * wave) + grp;
#pragma unroll
    for (int u = 0; u < N; ++u) {
        const int key = min(first + u * (H::TILES ? H::KPW : H::KPB), hi - 1);
        const int lp = page_of(a, key);
        const ch_u64 at = (ch_u64)(unsigned)sh.ids[p.page_off + lp - p.page_lo] * page_bytes + (unsigned)((key - lp * ps) * (2 * DH) + 16 * sub);
        dst[u] = stream16(kc + at);
        dst[N + u] = stream16(vc + at);
    }
    __builtin_amdgcn_sched_barrier(0);                       // (the addresses of further stages would take registers that are not there)
}

typedef __bf16 ch_v2b __attribute__((ext_vector_type(2)));
typedef float ch_v8f __attribute__((ext_vector_type(8)));
typedef short ch_v4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float dot2(unsigned a, unsigned b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(ch_v2b, a), __builtin_bit_cast(ch_v2b, b), c, false);
}

// A piece's cached keys, first stages sent ahead: the waves' softmax states (maximum in units of log 2, sum, weighted values) to `state`.
template <int GQ>
__device__ __forceinline__ void walk_piece(Args a, const Shared& sh, const Piece& p, Far kc, Far vc, int lane, int wave, uint4 (&ring)[kRing],
                                           const uint16_t* queries, uint16_t* tile, float* state) {
    using H = Heads<GQ>;
    a = again(a);
    lane = again_v(lane);
    const int hi = min(p.hi, p.pos), ns = (max(hi - p.lo, 0) + H::STEP - 1) / H::STEP;
    const float scale = a->scale * 1.4426950408889634f;      // scores in units of log 2
    auto walk = [&](auto take) {
        int left = ns, st = 0;
        while (left >= 2 * H::S) {
#pragma unroll
            for (int s = 0; s < H::S; ++s) {
                take(st + s, ring + s * H::SLOTS);
                __builtin_amdgcn_sched_barrier(0);
                send_keys<GQ>(a, sh, p, kc, vc, st + s + H::S, lane, wave, ring + s * H::SLOTS);
            }
            left -= H::S;
            st += H::S;
        }
        if (left > H::S) {
            const int more = left - H::S;
#pragma unroll
            for (int s = 0; s < H::S; ++s) {
                take(st + s, ring + s * H::SLOTS);
                __builtin_amdgcn_sched_barrier(0);
                if (s < more) send_keys<GQ>(a, sh, p, kc, vc, st + s + H::S, lane, wave, ring + s * H::SLOTS);
            }
            left -= H::S;
            st += H::S;
        }
#pragma unroll
        for (int s = 0; s < H::S; ++s)
            if (s < left) { take(st + s, ring + s * H::SLOTS); __builtin_amdgcn_sched_barrier(0); }
    };
    if constexpr (!H::TILES) {
        const int sub = lane % H::LPK, grp = lane / H::LPK, kb = p.lo + wave * H::KPW + grp;
        const uint4 q = *reinterpret_cast<const uint4*>(queries + sub * 8);
        float acc[8], m = -INFINITY, l = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = 0.f;
        walk([&](int stage, const uint4* at) {
            float w[H::U], mx = m;
#pragma unroll
            for (int u = 0; u < H::U; ++u) {
                float d = dot2((unsigned)again_v((int)q.x), at[u].x, 0.f);     // (not before this stage's turn: the sums of six would take registers)
                d = dot2(q.y, at[u].y, d);
                d = dot2(q.z, at[u].z, d);
                d = dot2(q.w, at[u].w, d);
                d = group_sum<H::LPK>(d) * scale;
                w[u] = kb + stage * H::STEP + u * H::KPB < hi ? d : -INFINITY;
                mx = fmaxf(mx, w[u]);
            }
            if (mx == -INFINITY) return;                     // this lane group has seen no key yet
            const float corr = __builtin_amdgcn_exp2f(m - mx);
            l *= corr;
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] *= corr;
#pragma unroll
            for (int u = 0; u < H::U; ++u) {
                float v[8];
                Vec16<bf16>::unpack(at[H::U + u], v);
                w[u] = __builtin_amdgcn_exp2f(w[u] - mx);
                l += w[u];
#pragma unroll
                for (int i = 0; i < 8; ++i) acc[i] = fmaf(w[u], v[i], acc[i]);
            }
            m = mx;
            // (now, not when the last stage's results are wanted: what is left undone of six stages takes registers)
            asm volatile("" : "+v"(m), "+v"(l), "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]), "+v"(acc[4]), "+v"(acc[5]), "+v"(acc[6]), "+v"(acc[7]));
        });
        // the lane groups: one maximum, then sums
        float mw = m;
#pragma unroll
        for (int o = H::LPK; o < 64; o <<= 1) mw = fmaxf(mw, lane_xor(mw, o));
        const float c = __builtin_amdgcn_exp2f(m - (mw == -INFINITY ? 0.f : mw));
        auto sum = [&](float v) { return swap_add<32>(swap_add<16>(dpp_add<0x128>(v))); };
        l = sum(l * c);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = sum(acc[i] * c);
        if (grp == 0) {
            float* const o = state + wave * H::STATE;
#pragma unroll
            for (int i = 0; i < 8; i += 4) *reinterpret_cast<float2*>(o + sub * 8 + i) = float2{acc[i], acc[i + 1]}, *reinterpret_cast<float2*>(o + sub * 8 + i + 2) = float2{acc[i + 2], acc[i + 3]};
            if (sub == 0) *reinterpret_cast<float2*>(o + DH) = float2{mw, l};
        }
    } else {
        // S^T = K Q^T and O^T = V^T P^T with v_mfma_f32_16x16x32_bf16 as in attn_decode_blocks.h: head lr is a column.
        constexpr int NC = DH / 32, ND = DH / 16, NV = H::NV, VS = H::VS, KPI = H::KPW;
        const int lr = lane & 15, lg = lane >> 4, key0 = lane / H::LPK, oct = lane % H::LPK;
        uint16_t* const mine = tile + wave * 32 * VS;
        ch_v8b q[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c)
            q[c] = ch_op(lr < GQ ? *reinterpret_cast<const uint4*>(queries + lr * DH + 32 * c + 8 * lg) : uint4{0, 0, 0, 0});
        ch_v4f acc[ND];
#pragma unroll
        for (int c = 0; c < ND; ++c) acc[c] = ch_v4f{0.f, 0.f, 0.f, 0.f};
        float m = -INFINITY, l = 0.f;
        walk([&](int stage, const uint4* at) {
            const int kt = p.lo + stage * H::STEP + 32 * wave;
            if (kt >= hi) return;                            // (uniform)
            const bool last = kt + 32 > hi;
            // (a wave's own part of LDS, served in order)
            auto stash = [&](const uint4* v, bool clean) {
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int i = 0; i < NV; ++i) {
                    const uint4 x = clean && kt + key0 + KPI * i >= hi ? uint4{0, 0, 0, 0} : v[i];       // weight 0, but 0 * infinity is NaN
                    *reinterpret_cast<uint4*>(mine + (key0 + KPI * i) * VS + oct * 8) = x;
                }
                __builtin_amdgcn_wave_barrier();
            };
            stash(at, false);
            ch_v4f sc[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                sc[h] = ch_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    sc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ch_op(*reinterpret_cast<const uint4*>(mine + (16 * h + lr) * VS + 32 * c + 8 * lg)), q[c], sc[h], 0, 0, 0);
            }
            stash(at + NV, last);
            float w[8], mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                w[e] = sc[e >> 2][e & 3] * scale;
                if (last && kt + 16 * (e >> 2) + 4 * lg + (e & 3) >= hi) w[e] = -INFINITY;
                mx = fmaxf(mx, w[e]);
            }
            mx = swap_max<16>(swap_max<32>(mx));
            if (__builtin_amdgcn_ballot_w64(mx > m)) {
                const float now = fmaxf(m, mx), corr = __builtin_amdgcn_exp2f(m - (now == -INFINITY ? 0.f : now));
                l *= corr;
                m = now;
#pragma unroll
                for (int c = 0; c < ND; ++c) acc[c] *= corr;
            }
            ch_v8f pf;
            const float base = m == -INFINITY ? 0.f : m;     // (no key of this head yet whose score is not -inf: weights 0)
#pragma unroll
            for (int e = 0; e < 8; ++e) { pf[e] = __builtin_amdgcn_exp2f(w[e] - base); l += pf[e]; }
            const ch_v8b pb = __builtin_convertvector(pf, ch_v8b);
            const uint16_t* const vrow = mine + (4 * lg + (lr >> 2)) * VS + 4 * (lr & 3);
#pragma unroll
            for (int c = 0; c < ND; ++c) {
                const ch_v4s lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ch_v4s __attribute__((address_space(3)))*)(vrow + 16 * c));
                const ch_v4s hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ch_v4s __attribute__((address_space(3)))*)(vrow + 16 * VS + 16 * c));
                acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ch_v8b, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7)), pb, acc[c], 0, 0, 0);
            }
        });
        l = swap_add<16>(swap_add<32>(l));
        if (lr < GQ) {
            float* const o = state + wave * H::STATE;
#pragma unroll
            for (int c = 0; c < ND; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[lr * DH + 16 * c + 4 * lg + e] = acc[c][e];
            if (lg == 0) *reinterpret_cast<float2*>(o + GQ * DH + 2 * lr) = float2{m, l};
        }
    }
}

// ---- the kernel -------------------------------------------------------------------------------------------------------------------
template <int GQ, int PQ, int PG, int RR>
__global__ void __launch_bounds__(kThreads)
decode_chain_kernel(const ChainArgs) {
    Args a = (Args)__builtin_amdgcn_kernarg_segment_ptr();
    using H = Heads<GQ>;
    extern __shared__ __align__(16) unsigned char ch_smem[];
    unsigned char* const rows = ch_smem;                                    // token rows [line of 64][row][128 bytes]; staged queries
    float* const red = reinterpret_cast<float*>(ch_smem + a->rows_bytes);    // partial results of the waves; their softmax states
    Shared& sh = *reinterpret_cast<Shared*>(ch_smem + a->rows_bytes + a->red_floats * 4);
    ChainEntry* const table = reinterpret_cast<ChainEntry*>(&sh + 1);
    uint16_t* const tile = reinterpret_cast<uint16_t*>(rows + kMaxPieces * 1024);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned* const joined = a->sync;
    unsigned* const frozen = a->sync + kCounters * kLineWords;

    // ---- who takes part: the blocks that run.  Normally all; after a millisecond those that have come by then, so that nobody
    // waits for a block that finds no room.
    if (wave == kStream) {
        const int c = (int)blockIdx.x % kCounters;
        unsigned mine = 0;
        if (lane == 0) mine = __hip_atomic_fetch_add(joined + c * kLineWords, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        mine = (unsigned)__builtin_amdgcn_readfirstlane((int)mine);
        int n = 0, rank = -1;
        if (!(mine & kClosed)) {
            const unsigned cap = lane < kCounters && lane < a->G ? (unsigned)(a->G - lane + kCounters - 1) / kCounters : 0u;
            const unsigned long long t0 = wall_clock64();
            bool closing = false;
            unsigned count = 0;
            while (true) {
                const unsigned v = lane < kCounters ? ld_far(joined + lane * kLineWords) : 0u;
                if (__all(v == cap)) { count = cap; break; }
                const unsigned f = lane < kCounters ? ld_far(frozen + lane * kLineWords) : 1u;
                if (__all(f != 0u)) { count = f - 1u; break; }
                const unsigned long long waited = wall_clock64() - t0;
                if (!closing && waited > kJoinTicks) {
                    unsigned here = lane < kCounters ? v & (kClosed - 1u) : 0u;
                    for (int o = 1; o < kCounters; o <<= 1) here += __shfl_xor(here, o);
                    const unsigned rounds = (unsigned)(a->G - 1) / max((unsigned)__builtin_amdgcn_readfirstlane((int)here), 1u);     // beyond the one that all together need
                    if (waited < (unsigned long long)rounds * max(kJoinTicks, kLayerTicks * (unsigned)a->n_entries)) continue;
                    closing = true;
                    if (lane < kCounters) {
                        const unsigned old = __hip_atomic_fetch_or(joined + lane * kLineWords, kClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        if (!(old & kClosed)) st_far(frozen + lane * kLineWords, (old & 0xffffu) + 1u);
                    }
                }
            }
            int sum = (int)count;                            // inclusive prefix over the counters
            for (int o = 1; o < kCounters; o <<= 1) {
                const int up = __shfl_up(sum, o);
                if (lane >= o && lane < kCounters) sum += up;
            }
            n = __shfl(sum, kCounters - 1);
            rank = __shfl(sum - (int)count, c) + (int)(mine & 0xffffu);
        }
        if (lane == 0) {
            sh.n = n; sh.rank = rank;
            sh.tries = a->tries;
        }
    } else if (wave == kStream + 1) {
        // the units of attention work, and how they are dealt
        const int T = a->T, nkv = a->nkv;
        const int pos = lane < T ? a->positions[lane] : 0;
        const int tiles = lane < T ? units_of(pos) : 0;
        int sum = tiles * nkv, longest = tiles;
        for (int o = 1; o < kChainMaxRows; o <<= 1) {
            const int up = __shfl_up(sum, o);
            if (lane >= o) sum += up;
        }
        for (int o = 1; o < kChainMaxRows; o <<= 1) longest = max(longest, __shfl_xor(longest, o));
        const int units = __shfl(sum, kChainMaxRows - 1);
        if (lane < kChainMaxRows) { sh.tiles[lane] = tiles; sh.before[lane + 1] = sum; }
        if (lane == 0) {
            sh.before[0] = 0;
            sh.direct = walks_whole_heads(T * nkv, a->G, longest, units);
            sh.workers = workers_of(sh.direct, T * nkv, units, a->G);
        }
    }
    __syncthreads();
    const int n = __builtin_amdgcn_readfirstlane(sh.n), rank = __builtin_amdgcn_readfirstlane(sh.rank);
    if (rank < 0) return;                                    // too late: the others do it all
    const int direct = __builtin_amdgcn_readfirstlane(sh.direct), workers = __builtin_amdgcn_readfirstlane(sh.workers);
    const bool planned = n >= a->G;                           // a block has one worker's pieces, the same in all layers
    if (planned && tid == 64 * kStream) plan_pieces(a, sh, rank);
    __syncthreads();
    auto load_ids = [&](int from, int step) {
        for (int i = 0; i < sh.n_pieces; ++i) {
            const Piece& p = sh.piece[i];
            const int* bt = a->tables + (size_t)a->token_req[p.row] * a->bt_stride + p.page_lo;
            const int np = page_of(a, p.hi - 1) - p.page_lo + 1;
            for (int k = from; k < np; k += step) sh.ids[p.page_off + k] = bt[k];
        }
    };
    if (planned) load_ids(tid, kThreads);
    for (int i = tid; i < (a->n_entries + 1) * (int)(sizeof(ChainEntry) / 8); i += kThreads) reinterpret_cast<ch_u64*>(table)[i] = reinterpret_cast<const ch_u64*>(a->entries)[i];
    __syncthreads();

    if (wave < kStream) {
        // ---- streaming waves ---------------------------------------------------------------------------------------------------------
        // A task's first loads go out before the rows are there, behind the results of the task before.
        auto product = [&](auto kind, auto groups, const ChainEntry* E) {
            constexpr int KIND = kind, RG = groups;
            for (int t = rank; t < tasks_of<KIND>(a); t += n) {
                uint4 ring[kRing];
                send_ahead<KIND, RG>(a, E, t, lane, wave, ring);
                meet();
                multiply<KIND, RG>(a, E, t, lane, wave, ring, rows, red);
                meet();
                meet();                                      // the results are on their way
            }
        };
        const int n_entries = a->n_entries;
        for (int e = 0; e < n_entries; ++e) {
            a = again(a);
            const ChainEntry* const E = table + e;
            product(std::integral_constant<int, QKV>{}, std::integral_constant<int, 2 * PQ>{}, E);
            for (int w = rank; w < workers; w += n) {
                if (!planned) { meet(); meet(); }            // the plan, its page ids
                const int np = __builtin_amdgcn_readfirstlane(sh.n_pieces);
                for (int i = 0; i < np; ++i) {
                    const Piece p = piece_of(sh, i);
                    const Far kc = uniform(E->k_cache), vc = uniform(E->v_cache);
                    const int hi = min(p.hi, p.pos);
                    uint4 ring[kRing];
#pragma unroll
                    for (int s = 0; s < H::S; ++s)
                        if (hi > p.lo + s * H::STEP) send_keys<GQ>(a, sh, p, kc, vc, s, lane, wave, ring + s * H::SLOTS);
                        else clear(ring + s * H::SLOTS, H::SLOTS);
                    if (i == 0) meet();                      // the queries
                    walk_piece<GQ>(a, sh, p, kc, vc, lane, wave, ring, reinterpret_cast<const uint16_t*>(rows + 1024 * i), tile, red + (i & 1) * kStream * H::STATE);
                    meet();
                }
                meet();                                      // the plan has been used, the results are on their way
            }
            product(std::integral_constant<int, OUT_PROJ>{}, std::integral_constant<int, RR>{}, E);
            product(std::integral_constant<int, GATE_UP>{}, std::integral_constant<int, 2 * PG>{}, E);
            product(std::integral_constant<int, DOWN>{}, std::integral_constant<int, RR>{}, E);
        }
        return;
    }

    // ---- control waves ----------------------------------------------------------------------------------------------------------------
    __builtin_amdgcn_s_setprio(2);
    const int cw = wave - kStream, ctid = tid - 64 * kStream;
    const int oi = lane & 7, om = lane >> 3;
    // Chunks of 1 KB, dealt over the control waves, to `rows` in order, again and again until no element in them is empty: what others write arrives so without a
    // further signal.  where(c): the lane's 16 bytes of chunk c.  Chunks from `halves` on hold `sums` float32 (some of the last 16 bytes may be nobody's).
    auto tries_left = [&]() { return *const_cast<const volatile int*>(&sh.tries); };
    auto give_up = [&]() {                                   // (known to the other blocks before anything that is computed from here on)
        if (tries_left() < 0) return;
        const Args b = again(a);
        st_far(b->sync + kGaveUp, 1u);
        if (b->gave_up) __hip_atomic_store(b->gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __threadfence_system();
        sh.tries = -1;
    };
    auto fetch = [&](int chunks, int halves, int sums, auto where) {
        ch_u64 open = cw < chunks ? ~0ull >> (64 - (chunks - cw + kControl - 1) / kControl) : 0ull;
        int tries = 0;
        while (open) {
            for (ch_u64 m = open; m; m &= m - 1) {
                const int c = cw + kControl * (int)__builtin_ctzll(m);
                __builtin_amdgcn_global_load_lds((ch_gptr)where(c), (ch_lptr)(rows + 1024 * c), 16, 0, kFarLoad);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            for (ch_u64 m = open; m; m &= m - 1) {
                const int k = (int)__builtin_ctzll(m), c = cw + kControl * k;
                const uint4 v = *reinterpret_cast<const uint4*>(rows + 1024 * c + 16 * lane);
                bool lacks;
                if (c < halves) lacks = (empty_halves(v.x) | empty_halves(v.y) | empty_halves(v.z) | empty_halves(v.w)) != 0;
                else {
                    const int left = sums - 4 * min(64 * (c - halves) + lane, (sums - 1) >> 2);
                    lacks = v.x == ~0u || (left > 1 && v.y == ~0u) || (left > 2 && v.z == ~0u) || (left > 3 && v.w == ~0u);
                }
                if (!__any(lacks)) open &= ~(1ull << k);
            }
            if (++tries > tries_left()) { give_up(); break; }
        }
    };
    // The rows [row][K] of a product, with ss the sums of squares [row][task] behind them.
    auto stage = [&](const unsigned char* src, int K, const unsigned char* ss) {
        const Args b = again(a);
        const int T = b->T, total = (K >> 6) * T * 8, magic = 65536 / T + 1;
        const int chunks = (total + 63) >> 6, sums = ss ? T * b->t_res : 0;
        fetch(chunks + ((sums + 255) >> 8), chunks, sums, [&](int c) -> const void* {
            if (c >= chunks) return ss + 16 * min(64 * (c - chunks) + lane, (sums - 1) >> 2);
            const int i = min(64 * c + lane, total - 1), row_line = i >> 3, line = (row_line * magic) >> 16, t = row_line - line * T;
            return src + 2 * (t * K + 64 * line + 8 * (i & 7));
        });
        meet();
    };
    auto row_factors = [&](int K, float eps) {               // (between the two meetings of a product)
        const Args b = again(a);
        const int T = b->T, parts = b->t_res;
        const float* const ss = reinterpret_cast<const float*>(rows + 1024 * (((K >> 6) * T * 8 + 63) >> 6));
        for (int t = cw; t < T; t += kControl) {
            float s = 0.f;
            for (int i = lane; i < parts; i += 64) s += ss[t * parts + i];
            s = wave_sum(s);
            if (lane == 0) sh.factor[t] = sh.tries < 0 ? __uint_as_float(0x7fc00000u) : rsqrtf(s / (float)K + eps);
        }
    };
    auto sum_of = [&](int out, int at) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < 2 * kStream; ++w) v += red[w * out + at];
        return v;
    };
    auto rounded = [&](float v) { return to_f32(from_f32<bf16>(v)); };

    // ---- O and down: into the residual stream, with the next norm's weight and sums of squares
    auto residual = [&](const unsigned char* src, int K, const float __attribute__((address_space(1)))* weight, bf16* y, float* ss, bool final_norm) {
        const Args b = again(a);
        const int T = b->T, d = b->d;
        for (int t = rank; t < b->t_res; t += n) {
            float x[RR], g[RR];
            bool mine[RR];
#pragma unroll
            for (int r = 0; r < RR; ++r) {
                const int col = t * b->cols + 8 * r + oi;
                mine[r] = cw == 0 && om < T && 8 * r + oi < b->cols && col < d;
                x[r] = mine[r] ? ld_far(b->x + (size_t)om * d + col) : 0.f;
                g[r] = mine[r] ? weight[col] : 0.f;
            }
            if (t == rank) stage(src, K, nullptr);
            else meet();
            meet();
            if (cw == 0) {
                float sq = 0.f;
                const float poison = sh.tries < 0 ? __uint_as_float(0x7fc00000u) : 0.f;
#pragma unroll
                for (int r = 0; r < RR; ++r) {
                    if (!mine[r]) continue;
                    const int col = t * b->cols + 8 * r + oi;
                    const float h = x[r] + b->rscale * rounded(sum_of(RR * 64, r * 64 + lane)) + poison;
                    put(y + (size_t)om * d + col, h * g[r]);
                    st_far(b->x + (size_t)om * d + col, h);
                    sq += h * h;
                }
#pragma unroll
                for (int o = 1; o < 8; o <<= 1) sq += lane_xor(sq, o);
                if (oi == 0) {
                    if (final_norm) {                        // [parts][16], for the product after the chain
                        put(ss + t * 16 + om, om < T ? sq : 0.f);
                        put(ss + t * 16 + 8 + om, 0.f);
                    } else if (om < T) put(ss + om * b->t_res + t, sq);
                }
            }
            meet();
        }
    };

    // Everything a phase needs is read from the arguments at its start.
#define CH_PHASE                                                                                     \
    const Args b = again(a);                                                                         \
    [[maybe_unused]] const ChainEntry* const E = table + e;                                          \
    [[maybe_unused]] const int T = b->T, d = b->d, nh = b->nh, nkv = b->nkv, ow = b->ow;             \
    unsigned char* const s = b->scratch + (size_t)e * b->at.stride
    const int n_entries = a->n_entries;
    for (int e = 0; e < n_entries; ++e) {
        // ---- QKV, rotary, cache write
        {
            CH_PHASE;
            for (int t = rank; t < b->t_qkv; t += n) {
                const int pair = t * PQ + cw, per_head = DH >> 4, head = pair / per_head, hj = 8 * (pair - head * per_head);
                const bool mine = cw < PQ && om < T && head < nh + 2 * nkv;
                int slot = -1;
                float c = 0.f, sn = 0.f;
                if (mine) {
                    slot = b->slots[om];
                    if (head < nh + nkv) {
                        const size_t at = (size_t)b->positions[om] * (DH >> 1) + hj + oi;
                        c = b->cos_t[at];
                        sn = b->sin_t[at];
                    }
                }
                if (t == rank) { stage(s + b->at.y_in, d, s + b->at.ss_in); row_factors(d, b->eps_in); }
                else meet();
                meet();
                if (mine) {
                    const float f = sh.factor[om];
                    float v0 = rounded(f * sum_of(PQ * 128, 2 * cw * 64 + lane)), v1 = rounded(f * sum_of(PQ * 128, (2 * cw + 1) * 64 + lane));
                    const bool value = head >= nh + nkv;
                    const int i0 = value ? 2 * hj + oi : hj + oi, i1 = value ? i0 + 8 : i0 + (DH >> 1);
                    if (!value) { const float r0 = v0 * c - v1 * sn; v1 = v0 * sn + v1 * c; v0 = r0; }
                    bf16* const near = head < nh ? (bf16*)(s + b->at.q) + ((size_t)om * nh + head) * DH
                                                 : (bf16*)(s + b->at.kv) + ((size_t)om * 2 * nkv + (head - nh)) * DH;
                    put(near + i0, v0);
                    put(near + i1, v1);
                    // For later steps; not of rows that are NaN because a wait was given up.
                    if (head >= nh && slot >= 0 && !(f != f && ld_far(b->sync + kGaveUp) != 0u)) {
                        const int page = slot / b->page_size, off = slot - page * b->page_size;
                        bf16 __attribute__((address_space(1)))* const plane = (bf16 __attribute__((address_space(1)))*)uniform(value ? E->v_cache : E->k_cache) + (((size_t)page * nkv + (head - nh - (value ? nkv : 0))) * b->page_size + off) * DH;
                        ((uint16_t __attribute__((address_space(1)))*)plane)[i0] = f32_to_bf16_bits(v0);
                        ((uint16_t __attribute__((address_space(1)))*)plane)[i1] = f32_to_bf16_bits(v1);
                    }
                }
                meet();
            }
        }

        // ---- attention
        for (int w = rank; w < workers; w += n) {
            CH_PHASE;
            if (!planned) {
                if (ctid == 0) plan_pieces(a, sh, w);
                meet();
                load_ids(ctid, 64 * kControl);
                meet();
            }
            const int np = __builtin_amdgcn_readfirstlane(sh.n_pieces);
            if (np > 0) {
                // the queries of a piece's heads, the new key and value
                fetch(np, np, 0, [&](int i) -> const void* {
                    const Piece p = piece_of(sh, i);
                    const int part = lane / H::LPK, at = lane % H::LPK * 8;
                    const bf16* const q = (const bf16*)(s + b->at.q) + ((size_t)p.row * nh + p.kvh * GQ) * DH + at;
                    const bf16* const kv = (const bf16*)(s + b->at.kv) + ((size_t)p.row * 2 * nkv + p.kvh) * DH + at;
                    return part < GQ || part > GQ + 1 || p.hi <= p.pos ? q + min(part, GQ - 1) * DH : part == GQ ? kv : kv + (size_t)nkv * DH;
                });
                meet();
                for (int i = 0; i < np; ++i) {               // the score of the step's own key, while the others are walked
                    const uint16_t* const at = reinterpret_cast<const uint16_t*>(rows + 1024 * i);
                    for (int j = cw; j < GQ; j += kControl) {
                        float d = bf16_bits_to_f32(at[j * DH + lane]) * bf16_bits_to_f32(at[GQ * DH + lane]);
                        d = wave_sum(d) * b->scale * 1.4426950408889634f;
                        if (lane == 0) sh.own[i][j] = d;
                    }
                }
                for (int i = 0; i < np; ++i) {
                    meet();                                  // the waves' states of piece i
                    const float* const st = red + (i & 1) * kStream * H::STATE;
                    const Piece p = piece_of(sh, i);
                    const bool own = p.hi > p.pos;
                    for (int x = ctid; x < GQ * DH; x += 64 * kControl) {
                        const int j = x / DH, c = x - j * DH;
                        float m = own ? sh.own[i][j] : -INFINITY, acc = 0.f, l = 0.f;
#pragma unroll
                        for (int v = 0; v < kStream; ++v) m = fmaxf(m, st[v * H::STATE + GQ * DH + 2 * j]);
                        const float base = m == -INFINITY ? 0.f : m;         // (every score is: all weights are 0, not exp2(-inf + inf))
#pragma unroll
                        for (int v = 0; v < kStream; ++v) {
                            const float k = __builtin_amdgcn_exp2f(st[v * H::STATE + GQ * DH + 2 * j] - base);
                            acc = fmaf(st[v * H::STATE + j * DH + c], k, acc);
                            l = fmaf(st[v * H::STATE + GQ * DH + 2 * j + 1], k, l);
                        }
                        if (own && sh.own[i][j] != -INFINITY) {
                            const float k = __builtin_amdgcn_exp2f(sh.own[i][j] - base);
                            acc = fmaf(bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(rows + 1024 * i)[(GQ + 1) * DH + c]), k, acc);
                            l += k;
                        }
                        if (direct) put((bf16*)(s + b->at.attn) + (size_t)p.row * ow + (size_t)(p.kvh * GQ + j) * DH + c, acc / l);
                        else {
                            put((float*)(s + b->at.acc) + ((size_t)p.slot * GQ + j) * DH + c, acc);
                            if (c < 2) put((float*)(s + b->at.ml) + ((size_t)p.slot * GQ + j) * 2 + c, c ? l : m);
                        }
                    }
                }
            }
            meet();
        }

        // ---- the pieces of a head together
        if (!direct && cw == 0) {
            CH_PHASE;
            constexpr int LP = DH / 4, GROUPS = 64 / LP, B = 4;              // lanes a piece, pieces at once, loads in flight
            const float* const p_acc = (const float*)(s + b->at.acc);
            const float* const p_ml = (const float*)(s + b->at.ml);
            const int c4 = 4 * (lane % LP), grp = lane / LP, units = sh.before[T];
            for (int hh = rank; hh < T * nh; hh += n) {
                const int row = hh / nh, h = hh - row * nh, kvh = h / GQ, j = h - kvh * GQ, seg = row * nkv + kvh;
                const int u0 = sh.before[row] + kvh * sh.tiles[row], u1 = u0 + sh.tiles[row] - 1;
                const int w0 = worker_of(u0, units, workers), w1 = worker_of(u1, units, workers);
                float m = -INFINITY, l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
                for (int first = w0; first <= w1; first += GROUPS * B) {     // (uniform)
                    const int w = first + grp;
                    float v[B][4], ml[B][2];
                    int tries = 0;
                    while (true) {
                        bool lacks = false;
#pragma unroll
                        for (int k = 0; k < B; ++k) {
                            const size_t at = (size_t)(seg + min(w + k * GROUPS, w1)) * GQ + j;
                            const ch_u64* const src = reinterpret_cast<const ch_u64*>(p_acc + at * DH + c4);
                            const ch_u64 x = ld_far(src), y = ld_far(src + 1), z = ld_far(reinterpret_cast<const ch_u64*>(p_ml + at * 2));
                            lacks |= (unsigned)x == ~0u || (unsigned)(x >> 32) == ~0u || (unsigned)y == ~0u || (unsigned)(y >> 32) == ~0u ||
                                     (unsigned)z == ~0u || (unsigned)(z >> 32) == ~0u;
                            v[k][0] = __uint_as_float((unsigned)x); v[k][1] = __uint_as_float((unsigned)(x >> 32));
                            v[k][2] = __uint_as_float((unsigned)y); v[k][3] = __uint_as_float((unsigned)(y >> 32));
                            ml[k][0] = __uint_as_float((unsigned)z); ml[k][1] = __uint_as_float((unsigned)(z >> 32));
                        }
                        if (!__any(lacks)) break;
                        if (++tries > tries_left()) { give_up(); break; }
                    }
                    float mx = m;
#pragma unroll
                    for (int k = 0; k < B; ++k) {
                        if (w + k * GROUPS > w1) ml[k][0] = -INFINITY;
                        mx = fmaxf(mx, ml[k][0]);
                    }
                    const float base = mx == -INFINITY ? 0.f : mx, corr = __builtin_amdgcn_exp2f(m - base);
                    l *= corr;
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] *= corr;
#pragma unroll
                    for (int k = 0; k < B; ++k) {
                        const float c = __builtin_amdgcn_exp2f(ml[k][0] - base);
                        l = fmaf(ml[k][1], c, l);
#pragma unroll
                        for (int i = 0; i < 4; ++i) acc[i] = fmaf(v[k][i], c, acc[i]);
                    }
                    m = mx;
                }
#pragma unroll
                for (int o = LP; o < 64; o <<= 1) {
                    const float mb = lane_xor(m, o), lb = lane_xor(l, o), mn = fmaxf(m, mb), base = mn == -INFINITY ? 0.f : mn;
                    const float ca = __builtin_amdgcn_exp2f(m - base), cb = __builtin_amdgcn_exp2f(mb - base);
                    l = fmaf(lb, cb, l * ca);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = fmaf(acc[i], ca, lane_xor(acc[i], o) * cb);
                    m = mn;
                }
                if (grp == 0) {
                    const float f = 1.f / l;
                    ch_u64 out = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) out |= (ch_u64)full_bits(acc[i] * f) << (16 * i);
                    st_far(reinterpret_cast<ch_u64*>((bf16*)(s + b->at.attn) + (size_t)row * ow + (size_t)h * DH + c4), out);
                }
            }
        }

        {
            CH_PHASE;
            residual(s + b->at.attn, ow, (const float __attribute__((address_space(1)))*)uniform(E->norm_mid), (bf16*)(s + b->at.y_mid), (float*)(s + b->at.ss_mid), false);
        }

        // ---- gate/up with the gated unit
        {
            CH_PHASE;
            for (int t = rank; t < b->t_gu; t += n) {
                if (t == rank) { stage(s + b->at.y_mid, d, s + b->at.ss_mid); row_factors(d, b->eps_mid); }
                else meet();
                meet();
                const int on = t * 8 * PG + 8 * cw + oi;
                if (cw < PG && om < T && on < b->di) {
                    const float f = sh.factor[om];
                    const float g = rounded(f * sum_of(PG * 128, cw * 64 + lane)), u = rounded(f * sum_of(PG * 128, (cw + PG) * 64 + lane));
                    put((bf16*)(s + b->at.act) + (size_t)om * b->di + on, silu_mul_fast(g, u));
                }
                meet();
            }
        }

        {
            CH_PHASE;
            const bool last = e + 1 == n_entries;
            unsigned char* const after = s + b->at.stride;
            residual(s + b->at.act, b->di, (const float __attribute__((address_space(1)))*)uniform(E[1].norm_in), last ? b->y_out : (bf16*)(after + b->at.y_in), last ? b->ss_out : (float*)(after + b->at.ss_in), last);
        }
    }
}

// x = embedding rows; the first norm half done (x times its weight, sums of squares in the first of the parts); nobody has joined the chain yet, and what its
// blocks hand on is empty: the first `handed` bytes of an entry's scratch, and all of it if heads are walked in pieces.
constexpr int kStartThreads = 1024;
__global__ void __launch_bounds__(kStartThreads)
chain_start_kernel(const int* __restrict__ tokens, const bf16* __restrict__ table, float scale, const float* __restrict__ weight, float* __restrict__ x,
                   unsigned char* scratch, Layout at, unsigned* __restrict__ sync, const int* __restrict__ positions, int d, int parts, int T, int nkv, int G, int n_entries) {
    __shared__ float red[16];
    const int t = blockIdx.x;
    bf16* const y = (bf16*)(scratch + at.y_in);
    float* const ss = (float*)(scratch + at.ss_in);
    if (t < T) {
        const bf16* row = table + (size_t)tokens[t] * d;
        float s = 0.f;
        for (int i = threadIdx.x; i < d; i += blockDim.x) {
            const float v = to_f32(row[i]) * scale;
            x[(size_t)t * d + i] = v;
            *(uint16_t*)(y + (size_t)t * d + i) = full_bits(v * weight[i]);
            s += v * v;
        }
        s = block_sum(s, red);
        for (int i = threadIdx.x; i < parts; i += blockDim.x) ss[t * parts + i] = i == 0 ? full_word(s) : 0.f;
        if (t == 0)
            for (int i = threadIdx.x; i < kSyncWords; i += blockDim.x) sync[i] = 0u;
        return;
    }
    int units = 0, longest = 0;
    for (int r = 0; r < T; ++r) { const int k = units_of(positions[r]); units += k * nkv; longest = max(longest, k); }
    const long long bytes = walks_whole_heads(T * nkv, G, longest, units) ? at.acc : at.stride;
    const uint4 ones{~0u, ~0u, ~0u, ~0u};
    for (int e = t - T; e < n_entries; e += (int)gridDim.x - T) {
        unsigned char* const to = scratch + (size_t)e * at.stride;
        for (long long i = (e ? 0 : at.q) + 16LL * threadIdx.x; i < bytes; i += 16 * kStartThreads) *reinterpret_cast<uint4*>(to + i) = ones;
    }
}

struct Plan { int pq, pg, rr, cols, t_qkv, t_res, t_gu; };

int per_unit(int items, int units) { return (items + units - 1) / units; }

Plan chain_plan(const ChainShape& s) {
    Plan p{};
    const int G = s.compute_units;
    if (G < 1) return p;
    const int pairs = (s.n_heads + 2 * s.n_kv_heads) * s.head_dim / 16, groups = per_unit(s.intermediate, 8);
    p.pq = per_unit(pairs, G);
    p.pg = per_unit(groups, G);
    p.cols = per_unit(s.hidden, G);
    p.rr = per_unit(p.cols, 8);
    p.t_qkv = per_unit(pairs, p.pq);
    p.t_gu = per_unit(groups, p.pg);
    p.t_res = per_unit(s.hidden, p.cols);
    return p;
}

inline long long up256(long long n) { return (n + 255) / 256 * 256; }

Layout chain_layout(const ChainShape& s, const Plan& p, int T) {
    Layout o{};
    long long at = 0;
    auto take = [&](long long bytes) { const long long was = at; at = up256(at + bytes); return was; };
    const long long d = s.hidden, ow = (long long)s.n_heads * s.head_dim, group = s.n_heads / s.n_kv_heads;
    const long long slots = ((long long)T * s.n_kv_heads + s.compute_units) * group;
    o.y_in = take(T * d * 2);
    o.ss_in = take((long long)T * p.t_res * 4);
    o.q = take(T * ow * 2);
    o.kv = take((long long)T * 2 * s.n_kv_heads * s.head_dim * 2);
    o.attn = take(T * ow * 2);
    o.y_mid = take(T * d * 2);
    o.ss_mid = take((long long)T * p.t_res * 4);
    o.act = take((long long)T * s.intermediate * 2);
    o.acc = take(slots * s.head_dim * 4);
    o.ml = take(slots * 2 * 4);
    o.stride = at;
    return o;
}

size_t lds_bytes(const ChainShape& s, const Plan& p, int T, int n_entries, int* rows_bytes, int* red_floats) {
    const int ow = s.n_heads * s.head_dim, group = s.n_heads / s.n_kv_heads;
    const int longest = std::max({s.hidden, ow, s.intermediate});
    const int rows = std::max((longest * T * 2 + 1023) / 1024 * 1024 + (T * p.t_res * 4 + 1023) / 1024 * 1024, kMaxPieces * 1024 + (group > 1 ? kStream * 32 * (s.head_dim + 8) * 2 : 0));
    const int red = std::max(2 * kStream * 64 * std::max({2 * p.pq, 2 * p.pg, p.rr}), 2 * kStream * group * (s.head_dim + 2));
    if (rows_bytes) *rows_bytes = rows;
    if (red_floats) *red_floats = red;
    return (size_t)rows + (size_t)red * 4 + sizeof(Shared) + (n_entries + 1) * sizeof(ChainEntry);
}

// Sizes that the kernel is built for: heads of 64 in groups of 1..4, and what a unit has of each product: one pair of row groups of QKV, two of gate/up and up to 8
// columns of the residual stream (up to 2,048 wide on 256 units), or two, three and 16 (up to 4,096 wide).
bool instance(const ChainShape& s, const Plan& p) {
    const int group = s.n_heads / s.n_kv_heads;
    return s.head_dim == DH && group >= 1 && group <= kMaxGroup && ((p.pq == 1 && p.pg == 2 && p.rr == 1) || (p.pq == 2 && p.pg == 3 && p.rr == 2));
}

// Up to here one launch is faster than the kernels one by one.  Rows are read by every block, so its advantage falls with them.  Speed of the kernels over its own at 40, 600,
// 2,000 keys and 2,000 beside 40: up to 2,048 wide (six shapes) 1.34..1.41, 1.26..1.32, 1.19..1.29 with one row, 1.04..1.12, 0.98..1.08, 1.02..1.11, 0.98..1.09 with eight (1.05 on average).
// Wider, groups of 1 and 2 (2,304 36:36, 4,096 40:40, 2,112 64:32): 1.24..1.25, 1.18..1.21, 1.20..1.22 with one row, 1.03..1.08, 1.04..1.08, 1.02..1.07, 1.01..1.05 with seven, 1.00..1.05, 0.99..1.03,
// 1.00..1.02, 0.98..1.00 with eight (0.96..0.98 with four to six of unlike lengths at one of them).  Groups of 3 and 4 (3,072 48:16, 2,304 64:16): 1.15..1.24, 1.11..1.17, 1.12..1.17; with five 1.08, 1.00..1.03, 1.04..1.07, 1.05..1.07, with six 1.03..1.06, 0.95..0.97, 1.01..1.03, 1.02..1.04,
// with seven 1.00..1.04, 0.92..0.94, 0.99..1.01, 0.99..1.00.
int most_rows(const ChainShape& s, const Plan& p) { return p.rr == 1 ? 8 : s.n_heads / s.n_kv_heads <= 2 ? 7 : 5; }
static_assert(kChainMaxRows >= 8, "rows of the narrow sizes");

template <int GQ, int PQ, int PG, int RR>
int go(const ChainArgs& a, int blocks, size_t lds, hipStream_t stream) {
    static bool raised[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return IC_ERR_UNSUPPORTED;
    if (!raised[dev]) {
        const hipError_t st = hipFuncSetAttribute((const void*)decode_chain_kernel<GQ, PQ, PG, RR>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (st != hipSuccess) { (void)hipGetLastError(); return (int)st; }
        raised[dev] = true;
    }
    hipLaunchKernelGGL((decode_chain_kernel<GQ, PQ, PG, RR>), dim3(blocks), dim3(kThreads), lds, stream, a);
    return ic_launch_status();
}

}  // namespace

int chain_supported(const ChainShape& s, int rows, int n_entries, int max_keys) {
    if (rows < 1 || rows > kChainMaxRows || s.compute_units < 64 || s.n_kv_heads < 1 || s.n_heads % s.n_kv_heads) return 0;
    if (s.hidden % 64 || s.intermediate % 64 || s.n_heads * s.head_dim % 64 || s.page_size < 16 || s.hidden > 16 * s.compute_units) return 0;
    if (2LL * 2 * s.intermediate * s.hidden > 0x7fffffffLL || 2LL * (s.n_heads + 2 * s.n_kv_heads) * s.head_dim * s.hidden > 0x7fffffffLL) return 0;
    if (2LL * s.n_kv_heads * s.page_size * s.head_dim > 0xffffffffLL) return 0;      // (a page's bytes are multiplied in 32 bits)
    const Plan p = chain_plan(s);
    if (!instance(s, p) || rows > most_rows(s, p) || p.t_res > ic_rule_sumsq_parts_max()) return 0;      // (the head product takes the row factors)
    const long long heads = (long long)rows * s.n_kv_heads, units = heads * ((max_keys + kUnit - 1) / kUnit);
    const long long keys = ((units + s.compute_units - 1) / s.compute_units + 6) * kUnit;
    const long long pieces = most_pieces(heads, units, s.compute_units);
    if (units * s.compute_units > 0x7fffffffLL || pieces > kMaxPieces || keys / s.page_size + 2 * pieces > kMaxPageIds) return 0;
    return lds_bytes(s, p, rows, n_entries, nullptr, nullptr) <= 160 * 1024;
}

int chain_sumsq_parts(const ChainShape& s) { return chain_plan(s).t_res; }

size_t chain_scratch_bytes(const ChainShape& s, int rows, int n_entries) {
    return (size_t)chain_layout(s, chain_plan(s), rows).stride * n_entries + kSyncWords * 4;
}

int chain_launch(const ChainShape& s, const ChainStep& st, int absent, hipStream_t stream) {
    const Plan p = chain_plan(s);
    ChainArgs a{st.entries, st.n_entries, st.rows, s.hidden, s.n_heads, s.n_kv_heads, s.intermediate, s.page_size, s.n_heads * s.head_dim, PageDivider(s.page_size)};
    a.scale = st.softmax_scale; a.rscale = st.residual_scale; a.eps_in = st.eps_in; a.eps_mid = st.eps_mid;
    a.positions = st.positions; a.slots = st.slots; a.token_req = st.token_req; a.tables = st.tables; a.bt_stride = st.table_stride;
    a.cos_t = st.cos_t; a.sin_t = st.sin_t; a.x = st.x;
    a.at = chain_layout(s, p, st.rows);
    a.sync = (unsigned*)st.scratch;
    a.scratch = (unsigned char*)st.scratch + kSyncWords * 4;
    a.gave_up = st.gave_up; a.tries = st.tries;
    a.y_out = (bf16*)st.y_out; a.ss_out = st.sumsq_out;
    a.G = s.compute_units; a.cols = p.cols; a.t_qkv = p.t_qkv; a.t_res = p.t_res; a.t_gu = p.t_gu;
    const size_t lds = lds_bytes(s, p, st.rows, st.n_entries, &a.rows_bytes, &a.red_floats);
    hipLaunchKernelGGL(chain_start_kernel, dim3(st.rows + st.n_entries), dim3(kStartThreads), 0, stream, st.tokens, (const bf16*)st.embed_table, st.embed_scale,
                       st.first_norm, st.x, a.scratch, a.at, a.sync, st.positions, s.hidden, p.t_res, st.rows, s.n_kv_heads, s.compute_units, st.n_entries);
    const int e = ic_launch_status();
    if (e) return e;
    const int group = s.n_heads / s.n_kv_heads;
#define CH_GO(GQ, PQ, PG, RR)                                                                                \
    if (group == GQ && p.pq == PQ && p.pg == PG && p.rr == RR) return go<GQ, PQ, PG, RR>(a, s.compute_units - absent, lds, stream)
    CH_GO(1, 1, 2, 1);
    CH_GO(2, 1, 2, 1);
    CH_GO(3, 1, 2, 1);
    CH_GO(4, 1, 2, 1);
    CH_GO(1, 2, 3, 2);
    CH_GO(2, 2, 3, 2);
    CH_GO(3, 2, 3, 2);
    CH_GO(4, 2, 3, 2);
#undef CH_GO
    return IC_ERR_UNSUPPORTED;
}

// The pieces of a step's attention as the kernel deals them, six ints each (worker, row, kv head, first key, key after the last, place), and for every (row, kv head)
// the workers from .. to whose pieces are brought together (from > to: none, a block walks the whole head): for tests.  Returns the number of pieces.
IC_EXPORT int ic_decode_chain_pieces(const int* positions, int rows, int kv_heads, int compute_units, int* pieces, int capacity, int* from_to) {
    if (!positions || rows < 1 || rows > kChainMaxRows || kv_heads < 1 || compute_units < 1) return IC_ERR_ARG;
    int tiles[kChainMaxRows], before[kChainMaxRows + 1] = {0}, longest = 0, n = 0;
    for (int r = 0; r < rows; ++r) {
        tiles[r] = units_of(positions[r]);
        before[r + 1] = before[r] + tiles[r] * kv_heads;
        longest = std::max(longest, tiles[r]);
    }
    const int units = before[rows], heads = rows * kv_heads;
    const bool whole = walks_whole_heads(heads, compute_units, longest, units);
    const int workers = workers_of(whole, heads, units, compute_units);
    for (int w = 0; w < compute_units; ++w)
        for_pieces(w, whole, workers, rows, kv_heads, positions, tiles, before, [&](int row, int kvh, int lo, int hi, int slot) {
            if (n < capacity && pieces) {
                int* const p = pieces + 6 * n;
                p[0] = w; p[1] = row; p[2] = kvh; p[3] = lo; p[4] = hi; p[5] = slot;
            }
            ++n;
        });
    for (int s = 0; from_to && s < heads; ++s) {
        const int row = s / kv_heads, u = before[row] + (s - row * kv_heads) * tiles[row];
        from_to[2 * s] = whole ? 1 : worker_of(u, units, workers);
        from_to[2 * s + 1] = whole ? 0 : worker_of(u + tiles[row] - 1, units, workers);
    }
    return n;
}
