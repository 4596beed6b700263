// Rows of float32 numbers as pairs of halves, as the products of pair_gemm.hip read them: what makes such rows (a pass of its own
// there, the norm before a product in ops.hip) shares this.
//
// A row of K numbers takes 4 bytes of each of round-up(K, 32): sixteen columns are 64 bytes, 32 of the halves h and 32 of the
// halves l.  `info` of a row is the power of two its numbers are scaled by and how many of them, scaled, are not small.
#pragma once
#include "common.h"
#include <limits.h>

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

#define PAIR_BIG 4.f            // scaled numbers of this size and more are big

// N scaled numbers as two planes of N halves; T: the type of N halves.
template <typename T>
__device__ __forceinline__ void pair_up(const float* v, T& h, T& l) {
    constexpr int N = sizeof(T) / 2;
    typedef _Float16 halves __attribute__((ext_vector_type(N)));
    halves hv, lv;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        hv[i] = static_cast<_Float16>(v[i]);
        lv[i] = static_cast<_Float16>((v[i] - static_cast<float>(hv[i])) * 4096.f);
    }
    h = __builtin_bit_cast(T, hv);
    l = __builtin_bit_cast(T, lv);
}

// From the bits of a row's largest magnitude: the power of two that brings it to 2^14 .. 2^15.
__device__ __forceinline__ int pair_scale(uint32_t top) {
    return top == 0 || top >= 0x7f800000u ? 0 : 14 - ilogbf(__uint_as_float(top));
}

// Where in a row's bytes the half h of column k lies; its l is 32 bytes behind.
__device__ __forceinline__ int pair_place(int k) { return (k >> 4) * 64 + (k & 15) * 2; }

__device__ __forceinline__ int2 pair_row_info(int scale, uint32_t top, int big) {
    return make_int2(scale, top == 0 ? INT_MAX : top >= 0x7f800000u ? -1 : big);
}
