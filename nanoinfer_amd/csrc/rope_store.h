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

    template <int V> struct Angles { float c[V], s[V]; };

    __device__ __forceinline__ bool rotates(int head) const { return head < H + KVH; }

    // what dims d to d + V of a head are rotated by at a position
    template <int V> __device__ __forceinline__ Angles<V> angles(int pos, int d) const {
        Angles<V> t;
        VecIO<float, V>::load(cos_t + static_cast<size_t>(pos) * (hd / 2) + d, t.c);
        VecIO<float, V>::load(sin_t + static_cast<size_t>(pos) * (hd / 2) + d, t.s);
        return t;
    }

    // where head `head` (queries', then keys', then values') of row m goes, null where it is not stored
    __device__ __forceinline__ bf16_t* place(int m, int slot, int head) const {
        if (head < H) return q + (static_cast<size_t>(m) * H + head) * hd;
        if (slot < 0) return nullptr;
        const int g = head < H + KVH ? head - H : head - H - KVH, page = slot / page_size;
        return (head < H + KVH ? kpool : vpool) + ((static_cast<size_t>(page) * KVH + g) * page_size + (slot - page * page_size)) * hd;
    }

    // V neighbouring dims from dim d < hd / 2 on, and the V half a head behind them, to the head's place
    template <int V> __device__ __forceinline__ void turned(bf16_t* to, int d, const float* a, const float* b, const Angles<V>& t) const {
        float first[V], second[V];
#pragma unroll
        for (int e = 0; e < V; ++e) {
            first[e] = a[e] * t.c[e] - b[e] * t.s[e];
            second[e] = a[e] * t.s[e] + b[e] * t.c[e];
        }
        store_packed<bf16_t, V>(to + d, first);
        store_packed<bf16_t, V>(to + d + hd / 2, second);
    }

    template <int V> __device__ __forceinline__ void plain(bf16_t* to, int d, const float* a, const float* b) const {
        store_packed<bf16_t, V>(to + d, a);
        store_packed<bf16_t, V>(to + d + hd / 2, b);
    }
};
