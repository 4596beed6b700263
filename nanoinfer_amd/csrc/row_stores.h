// Stores of a tile's rows.  The sums of a block of 16 x 16 lie so that lane l has four neighbouring columns (lane group l / 16) of row l % 16:
// one store of a wavefront is then 64 bytes of each of sixteen rows, half a line.  Two blocks side by side exchange halves before they go
// out, and a store is 128 bytes of each of eight rows.  Measured on products that end with all their results at once, to float32:
// wide_gemm.hip, 2,045 rows on [2048, 2048], 22.7 -> 20.6 us.  (Not in pair_gemm.hip, whose results are worked out on the way: a float32
// prompt of 1,700 tokens 15.29 -> 15.45 ms.)
#pragma once
#include "common.h"

// Lanes 0 to 7 and 8 to 15 of every sixteen hold a and b of rows r and r + 8: afterwards all of them a part of row r in a (the lower lanes a's,
// the upper ones b's) and of row r + 8 in b.  All lanes have to come here.
template <typename V> __device__ __forceinline__ void rows_together(V& a, V& b, bool upper) {
    uint32_t* pa = reinterpret_cast<uint32_t*>(&a);
    uint32_t* pb = reinterpret_cast<uint32_t*>(&b);
#pragma unroll
    for (int e = 0; e < static_cast<int>(sizeof(V) / 4); ++e) {
        const uint32_t t = upper ? pa[e] : pb[e];
        const uint32_t other = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(static_cast<int>(t), static_cast<int>(t), 0x128, 0xf, 0xf, false));   // row_ror:8
        pa[e] = upper ? other : pa[e];
        pb[e] = upper ? pb[e] : other;
    }
}
