// A float32 number as the sum of three bfloat16 numbers, for the float32 kernels that multiply on the bfloat16 matrix cores: the nearest one, the one nearest
// to what is left, and the rest, which has 7 bits at most; every subtraction is exact (finite values that do not round to infinity).  A second part is at most
// 2^-8 of its number, a third 2^-17, of either sign: the products that are left out (below) are 2^-24.2 of a product at most and nothing on average.  With the upper
// 16 bits as the first part (no rounding, the same number of instructions) they all had the product's sign: 2^-24.5 on average, up to 2^-21.2.  The conversion takes
// no longer in gemm_f32.hip; attention takes 1.7 % longer with it (101 forms; 2,048 tokens of 24:8 heads of 64 87 -> 93 us, of 32:8 heads of 128 225 -> 231).
#pragma once
#include "common.h"
#include <type_traits>
#include <utility>

typedef float parts_v4f __attribute__((ext_vector_type(4)));
typedef unsigned parts_v4u __attribute__((ext_vector_type(4)));
typedef __bf16 parts_v8b __attribute__((ext_vector_type(8)));
typedef float parts_v2f __attribute__((ext_vector_type(2)));
typedef __bf16 parts_v2b __attribute__((ext_vector_type(2)));

template <typename F, int... Is> __device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void each(F&& f) { each_of(f, std::make_integer_sequence<int, N>{}); }

// Four values in three bfloat16 parts each: step O of 22 (level O / 10: the values are rounded in pairs, then that is taken off), one instruction each.
struct Split4 {
    float y[4], t[4];
    unsigned p[3][2];
};
// BY_HAND: the conversion as assembly, for products written as assembly too (of the other the compiler makes bfloat16 vectors there, which it takes apart and copies until
// the large shapes spill).  It knows neither conversion nor product then, and two wait states belong between them: other instructions, which the caller sees to.
template <int O, bool BY_HAND = false> __device__ __forceinline__ void split_step(Split4& s) {
    constexpr int L = O / 10, Q = O % 10;
    if constexpr (Q < 2 && BY_HAND) asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(s.p[L][Q]) : "v"(s.y[2 * Q]), "v"(s.y[2 * Q + 1]));
    else if constexpr (Q < 2) s.p[L][Q] = __builtin_bit_cast(unsigned, __builtin_convertvector(parts_v2f{s.y[2 * Q], s.y[2 * Q + 1]}, parts_v2b));
    else if constexpr (Q < 6) s.t[Q - 2] = __uint_as_float(Q % 2 ? s.p[L][(Q - 2) / 2] & 0xffff0000u : s.p[L][(Q - 2) / 2] << 16);
    else s.y[Q - 6] -= s.t[Q - 6];
}
constexpr int kSplitSteps = 22;

// The six of the nine products of parts that count, the small ones first: part X of one factor times part Y of the other.
constexpr int kPartTerms = 6;
constexpr int kPartX[kPartTerms] = {2, 0, 1, 1, 0, 0}, kPartY[kPartTerms] = {0, 2, 1, 0, 1, 0};

// Where a result has to be computed again with the float32 instructions: what is not finite has no parts (inf - inf), and parts under 2^-126 are subnormal bfloat16 numbers, or
// nothing, so that numbers under 2^-102 are no longer the sum of theirs (2^-21 off at 2^-113).  These show by their results: under 2^-64 and not 0.
// One multiply-add, one shift with an add and one minimum a result (as comparisons of each: 2 % of a product's time, 3 % of attention's).
struct PartsCheck {
    float t = 0.f;                   // 0, or not a number
    unsigned least = ~0u;            // of twice the bits (no sign), less 1: 0 comes last
    __device__ __forceinline__ void add(float x) {
        t = fmaf(x, 0.f, t);
        least = min(least, (__float_as_uint(x) << 1) - 1u);
    }
    __device__ __forceinline__ bool failed() const { return !(t == 0.f) || least < 2u * 0x1f800000u - 1u; }    // (the bits of 2^-64)
};
