// A float32 number as the sum of three bfloat16 numbers, for the float32 kernels that multiply on the bfloat16 matrix cores: its upper 16 bits, those of
// what is left, and the rest, which has 8 bits at most; every subtraction is exact (normal, finite values).
#pragma once
#include "common.h"
#include <type_traits>
#include <utility>

typedef float parts_v4f __attribute__((ext_vector_type(4)));
typedef unsigned parts_v4u __attribute__((ext_vector_type(4)));
typedef __bf16 parts_v8b __attribute__((ext_vector_type(8)));

template <typename F, int... Is> __device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void each(F&& f) { each_of(f, std::make_integer_sequence<int, N>{}); }

// Four values in three bfloat16 parts each: step O of 22 (level O / 10: the parts' upper halves are packed, then taken off).
struct Split4 {
    float y[4], t[4];
    unsigned p[3][2];
};
template <int O> __device__ __forceinline__ void split_step(Split4& s) {
    constexpr int L = O / 10, Q = O % 10;
    if constexpr (Q < 2) s.p[L][Q] = __builtin_amdgcn_perm(__float_as_uint(s.y[2 * Q + 1]), __float_as_uint(s.y[2 * Q]), 0x07060302);
    else if constexpr (Q < 6) s.t[Q - 2] = __uint_as_float(__float_as_uint(s.y[Q - 2]) & 0xffff0000u);
    else s.y[Q - 6] -= s.t[Q - 6];
}
constexpr int kSplitSteps = 22;

// The six of the nine products of parts that count, the small ones first: part X of one factor times part Y of the other.
constexpr int kPartTerms = 6;
constexpr int kPartX[kPartTerms] = {2, 0, 1, 1, 0, 0}, kPartY[kPartTerms] = {0, 2, 1, 0, 1, 0};
