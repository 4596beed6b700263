// An RMSNorm between two products of many rows, in two halves: the product onto the residual stream leaves h * weight in the compute
// type and the sums of h^2 over 64 columns at a time, and the product behind the norm divides its rows by their root mean squares.
// RMSNorm(h) . W^T = ((h * weight) . W^T) / rms(h), row by row: every element of the operand is rounded once either way, and the addend
// of the stream is not rounded at all.  A norm of its own reads the product's result and the stream and writes both again, 49 MB for
// 1,999 rows of 2,048, 11 us at the rate of a copy; in the product's epilogue 16 MB less pass, behind stores that no other work hides.
// Measured (us, product and norm : this): 1,999 rows on [2048, 2048] 29.5 : 23.7, on [2048, 8192] 73.3 : 66.3, 1,100 on [2048, 2048]
// 24.3 : 21.6; the product behind, [16384, 2048] with SwiGLU, 109.5 -> 112 for its rows' factors (two rounds of workgroups, each with
// its sums of 32 parts a row to load first).  A prompt of 1,999 tokens of the 1B shape 4,573 -> 4,472 us.
#pragma once
#include "common.h"

// What a product does with the residual stream in its epilogue: h += product, and where `next` is set next = h * weight and the sums of squares.
struct StreamStore {
    float* h;               // [M, N]
    const float* weight;    // [N], the next norm's
    bf16_t* next;           // [M, N], null: nothing is left
    float* ss;              // [M, N / 64]
};

// What the product behind such a norm is given beside its rows.
struct RowNorm {
    const float* ss;        // [M, parts]
    int parts;              // a multiple of four, at most 64
    float eps;
};

// The share that thread `tid` of THREADS has in the sum of squares of one of ROWS rows from m0 on; asked for before the operands.  With 60 parts and
// more the compiler adds up in the branch of the last vector, and the first operands wait for that; without branches (a part that is not there
// loaded again, counted as zeros) it does not, and is no faster: 1,999 rows on [28672, 4096], 64 parts, 381 us so and 383 without, on [16384, 2048], 32
// parts, 112.7 and 113.5.
template <int ROWS, int THREADS> struct RowSquares {
    static constexpr int EACH = THREADS / ROWS, LOADS = 16 / EACH;      // threads a row; 64 parts in vectors of four
    static_assert(THREADS % ROWS == 0 && 16 % EACH == 0, "whole threads a row");
    float4 v[LOADS];

    __device__ __forceinline__ void ask(const RowNorm& norm, int m0, int M, int tid) {
        const float* row = norm.ss + static_cast<size_t>(min(m0 + tid / EACH, M - 1)) * norm.parts;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int p = (tid % EACH + i * EACH) * 4;
            v[i] = p < norm.parts ? *reinterpret_cast<const float4*>(row + p) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }

    // 1 / rms of the row, in all of its threads
    __device__ __forceinline__ float factor(const RowNorm& norm, int K) const {
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) sum += (v[i].x + v[i].y) + (v[i].z + v[i].w);
#pragma unroll
        for (int off = 1; off < EACH; off <<= 1) sum += __shfl_xor(sum, off, WAVE);
        return 1.f / sqrtf(sum / static_cast<float>(K) + norm.eps);
    }
};
