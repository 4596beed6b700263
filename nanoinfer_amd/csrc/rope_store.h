// What the products of many rows with the stacked matrix [q; k; v] do with a result in their epilogue: queries and keys are rotated
// over the whole head, queries go to rows of their own, keys and values into the cache's pages.
#pragma once
#include "common.h"

struct RopeStore {
    const int32_t* positions;    // [M]
    const float *cos_t, *sin_t;  // [positions, hd / 2]
    const int32_t* slots;        // [M]: place in the pools, below zero: not stored; null: none is
    bf16_t* q;                   // [M, H * hd]
    bf16_t *kpool, *vpool;       // [pages, KVH, page_size, hd]
    int H, KVH, hd, page_size;

    // V neighbouring dims of head `head` (queries', then keys', then values') of row m from dim d < hd / 2 on, and the V half a head behind them
    template <int V> __device__ __forceinline__ void put(int m, int pos, int slot, int head, int d, const float* a, const float* b) const {
        const int half = hd / 2;
        bf16_t* to;
        if (head < H) {
            to = q + (static_cast<size_t>(m) * H + head) * hd;
        } else {
            if (slot < 0) return;
            const int g = head < H + KVH ? head - H : head - H - KVH, page = slot / page_size;
            to = (head < H + KVH ? kpool : vpool) + ((static_cast<size_t>(page) * KVH + g) * page_size + (slot - page * page_size)) * hd;
        }
        if (head < H + KVH) {
            float c[V], s[V], first[V], second[V];
            VecIO<float, V>::load(cos_t + static_cast<size_t>(pos) * half + d, c);
            VecIO<float, V>::load(sin_t + static_cast<size_t>(pos) * half + d, s);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                first[e] = a[e] * c[e] - b[e] * s[e];
                second[e] = a[e] * s[e] + b[e] * c[e];
            }
            store_packed<bf16_t, V>(to + d, first);
            store_packed<bf16_t, V>(to + d + half, second);
        } else {
            store_packed<bf16_t, V>(to + d, a);
            store_packed<bf16_t, V>(to + d + half, b);
        }
    }
};
