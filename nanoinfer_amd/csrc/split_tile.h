// The tile of a float32 product by six bfloat16 products of the operands' three parts each (tile_gemm.hip says why), for the
// kernels that make it: of whole products, and of the tiles that pair_gemm.hip leaves.
#pragma once
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx16_t __attribute__((ext_vector_type(16)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

#define TG_XCDS 8

// Workgroups are dealt to the eight XCDs in turn; this gives each XCD a run of neighbouring tiles, so that the
// workgroups that read the same rows of W find them in one L2.
__device__ __forceinline__ int tile_of_block(int id, int total) {
    const int q = total / TG_XCDS, r = total % TG_XCDS, xcd = id % TG_XCDS, slot = id / TG_XCDS;
    return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
}

// The float32 numbers a and b multiplied and added up one after the other, in 64 bits; NaN is its own end.
__device__ __forceinline__ float plain_dot(const float* __restrict__ a, const float* __restrict__ b, int count) {
    double s = 0.0;
#pragma nounroll
    for (int k = 0; k < count && s == s; k += 4) {
        const float4 u = *reinterpret_cast<const float4*>(a + k), v = *reinterpret_cast<const float4*>(b + k);
        s += static_cast<double>(u.x) * v.x;
        s += static_cast<double>(u.y) * v.y;
        s += static_cast<double>(u.z) * v.z;
        s += static_cast<double>(u.w) * v.w;
    }
    return static_cast<float>(s);
}

// Four float32 numbers as three times four bfloat16 numbers that add up to them.
__device__ __forceinline__ void split3(const float4 a, uint2& h, uint2& m, uint2& l) {
    const float v[4] = {a.x, a.y, a.z, a.w};
    uint32_t hw[2], mw[2], lw[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        hw[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
        const float r0 = v[2 * i] - __uint_as_float(hw[i] << 16);
        const float r1 = v[2 * i + 1] - __uint_as_float(hw[i] & 0xffff0000u);
        mw[i] = pack_bf16x2(r0, r1);
        lw[i] = pack_bf16x2(r0 - __uint_as_float(mw[i] << 16), r1 - __uint_as_float(mw[i] & 0xffff0000u));
    }
    h = make_uint2(hw[0], hw[1]);
    m = make_uint2(mw[0], mw[1]);
    l = make_uint2(lw[0], lw[1]);
}

// What a workgroup's operands wait for.  AHEAD: the operands of a slab are read from LDS while the slab before is
// multiplied, in a second set of registers (a product of 32 workgroups 121 -> 113 us); the largest tile has no room for
// that set and reads them when their slab begins.
enum { TG_STORE = 0, TG_GATED = 1, TG_ROPE = 2, TG_STREAM = 3 };       // the last two: products of bfloat16 rows alone (rope_store.h, row_norm.h)

// EPI TG_STORE: out[share][m][n] (shares > 1: float32 sums of every share).  TG_GATED: W is [gate; up] stacked, N its
// rows; blocks of 32 columns of a tile come from the two halves in turn, so that a lane holds gate and up of the same
// output; out[m][n] = act(gate) * up, N / 2 wide.
//
// GROUPED: the rows of x belong to groups (the tokens of one expert each), every group has N rows of W of its own.  The
// rows of group e stand at the places offsets[e] .. offsets[e + 1] - 1; place p takes row rows[p] of x (rows null: row p).
// No tile spans two groups.  How many tiles the groups need is known on the device alone: the grid is the most that so
// many rows in so many groups can need, and a workgroup without a tile ends at once.
struct Groups {
    const int32_t* offsets;      // [count + 1]
    const int32_t* rows;         // [places], or null
    int count;
    size_t wstride;              // numbers from one group's rows of W to the next group's
    int ldw;                     // numbers from one row of W to the next
};

// Two slabs in LDS: a row takes SPLIT_ROWB bytes, the rows of x and of W of a slab stand apart.
#define SPLIT_ROWB (3 * 16 * 2 + 16)
template <int BM, int BN> struct SplitLds { static constexpr int BYTES = 2 * (BM + BN) * SPLIT_ROWB; };
struct SplitSlabs {
    char *x[2], *w[2];
    template <int BM, int BN> static __device__ __forceinline__ SplitSlabs in(char* lds) {      // SplitLds<BM, BN>::BYTES
        constexpr int SLAB = (BM + BN) * SPLIT_ROWB;
        return SplitSlabs{{lds, lds + SLAB}, {lds + BM * SPLIT_ROWB, lds + SLAB + BM * SPLIT_ROWB}};
    }
};

// The tile whose first row (place) is m0 and whose columns are the nt-th BN, over the K range kbeg to kend of share `share`.
// M: one behind the last row of the tile's group; K: numbers from one row of x to the next.
template <int BM, int BN, int WM, int WN, bool AHEAD, int EPI, bool GROUPED>
__device__ __forceinline__ void split_tile(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ out, int M, int N,
                                           int K, int m0, int nt, int share, int kbeg, int kend, int ldw, const int32_t* __restrict__ rows,
                                           const GatedUnit& act, const SplitSlabs& slabs) {
    constexpr int THREADS = WM * WN * WAVE;
    constexpr int BK = 16;
    constexpr int ROWB = SPLIT_ROWB;
    constexpr int TMB = BM / WM / 32, TNB = BN / WN / 32;
    constexpr int CPR = BK / 4;                         // chunks of four numbers a row
    constexpr int CA = BM * CPR / THREADS, CB = BN * CPR / THREADS, CH = CA + CB;
    static_assert(BM * CPR % THREADS == 0 && BN * CPR % THREADS == 0, "whole chunks a thread");
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const int half = N / 2;

    const float* src[CH];
    int dst[CH];
    const int kc = (tid % CPR) * 4;                     // the same for all chunks of a thread
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const bool isx = c < CA;
        const int r = (tid + (isx ? c : c - CA) * THREADS) / CPR;
        if (isx) {
            int row = min(m0 + r, M - 1);
            if constexpr (GROUPED)
                if (rows) row = rows[row];
            src[c] = x + static_cast<size_t>(row) * K;
            dst[c] = r * ROWB + kc * 2;
        } else {
            int n;
            if constexpr (EPI == TG_GATED) {
                const int n_out = min(nt * (BN / 2) + (r / 64) * 32 + (r & 31), half - 1);
                n = ((r >> 5) & 1) * half + n_out;
            } else {
                n = min(nt * BN + r, N - 1);
            }
            src[c] = w + static_cast<size_t>(n) * ldw;
            dst[c] = r * ROWB + kc * 2;
        }
    }
    struct Raw { float4 v[CH]; };
    struct Frags { bf16x8_t a[3][TMB], b[3][TNB]; };
    auto fetch = [&](Raw& s, int k0) {
        const int k = k0 + kc < kend ? k0 + kc : kbeg;   // a chunk is inside a share or outside it
#pragma unroll
        for (int c = 0; c < CH; ++c) s.v[c] = *reinterpret_cast<const float4*>(src[c] + k);
    };
    auto put = [&](const Raw& s, int c, int buf, int k0) {
        uint2 h, m, l;
        split3(s.v[c], h, m, l);
        if (k0 + kc >= kend) h = m = l = make_uint2(0, 0);
        char* p = (c < CA ? slabs.x[buf] : slabs.w[buf]) + dst[c];
        *reinterpret_cast<uint2*>(p) = h;
        *reinterpret_cast<uint2*>(p + BK * 2) = m;
        *reinterpret_cast<uint2*>(p + BK * 4) = l;
    };
    const int wm = wave / WN, wn = wave % WN;
    const int aoff = (wm * (BM / WM) + (lane & 31)) * ROWB + (lane >> 5) * 16;
    const int boff = (wn * (BN / WN) + (lane & 31)) * ROWB + (lane >> 5) * 16;
    auto read = [&](Frags& f, int buf) {
#pragma unroll
        for (int p = 2; p >= 0; --p) {
#pragma unroll
            for (int i = 0; i < TMB; ++i) f.a[p][i] = *reinterpret_cast<const bf16x8_t*>(slabs.x[buf] + aoff + 32 * i * ROWB + p * BK * 2);
#pragma unroll
            for (int j = 0; j < TNB; ++j) f.b[p][j] = *reinterpret_cast<const bf16x8_t*>(slabs.w[buf] + boff + 32 * j * ROWB + p * BK * 2);
        }
    };
    floatx16_t acc[TMB][TNB];
#pragma unroll
    for (int i = 0; i < TMB; ++i)
#pragma unroll
        for (int j = 0; j < TNB; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    // one slab: its operands are in registers; the next slab's are read, the one behind that is taken apart and written
    auto step = [&](int k0, const Frags& now, Frags& next, Raw& raw, int rd, int wr) {
        if constexpr (AHEAD) read(next, rd);
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};      // the small products first
#pragma unroll
        for (int g = 0; g < 6; ++g) {
#pragma unroll
            for (int i = 0; i < TMB; ++i)
#pragma unroll
                for (int j = 0; j < TNB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(now.a[PA[g]][i], now.b[PB[g]][j], acc[i][j], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < CH; ++c)
                if (c >= g * CH / 6 && c < (g + 1) * CH / 6) put(raw, c, wr, k0 + 2 * BK);
        }
        fetch(raw, k0 + 4 * BK);
        // a matrix instruction occupies its pipe for 32 cycles: room for a read, three vector instructions and a write
#pragma unroll
        for (int g = 0; g < 6 * TMB * TNB; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
        __syncthreads();
    };
    Raw r0, r1;
    Frags f0, f1;
    fetch(r0, kbeg);
    fetch(r1, kbeg + BK);
#pragma unroll
    for (int c = 0; c < CH; ++c) put(r0, c, 0, kbeg);
    if constexpr (AHEAD) {
#pragma unroll
        for (int c = 0; c < CH; ++c) put(r1, c, 1, kbeg + BK);
        fetch(r0, kbeg + 2 * BK);
        fetch(r1, kbeg + 3 * BK);
    } else {
        fetch(r0, kbeg + 2 * BK);
    }
    __syncthreads();
    if constexpr (AHEAD) {
        read(f0, 0);
        __syncthreads();
        for (int k0 = kbeg; k0 < kend; k0 += 2 * BK) {      // (a slab past the end is zeros)
            step(k0, f0, f1, r0, 1, 0);
            step(k0 + BK, f1, f0, r1, 0, 1);
        }
    } else {
        for (int k0 = kbeg; k0 < kend; k0 += 2 * BK) {
            read(f0, 0);
            step(k0 - BK, f0, f0, r1, 0, 1);
            read(f0, 1);
            step(k0, f0, f0, r0, 0, 0);
        }
    }

    const int cols = EPI == TG_GATED ? half : N;
    float* base = out + static_cast<size_t>(share) * M * cols;
    auto row_of = [&](int i, int e) { return m0 + wm * (BM / WM) + 32 * i + 8 * (e / 4) + 4 * (lane >> 5) + (e & 3); };
    float zero = 0.f;                // NaN once a number that this lane holds is not finite
#pragma unroll
    for (int i = 0; i < TMB; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int m = row_of(i, e);
            if (m >= M) continue;
            if constexpr (EPI == TG_GATED) {
#pragma unroll
                for (int j = 0; j < TNB / 2; ++j) {
                    const int n = nt * (BN / 2) + wn * (BN / WN / 2) + 32 * j + (lane & 31);
                    if (n < cols) base[static_cast<size_t>(m) * cols + n] = act.value(acc[i][2 * j][e], acc[i][2 * j + 1][e]);
                }
            } else {
#pragma unroll
                for (int j = 0; j < TNB; ++j) {
                    const int n = nt * BN + wn * (BN / WN) + 32 * j + (lane & 31);
                    if (n < cols) base[static_cast<size_t>(m) * cols + n] = act.plain(acc[i][j][e]);
                }
            }
#pragma unroll
            for (int j = 0; j < TNB; ++j) zero = fmaf(acc[i][j][e], 0.f, zero);
        }
    }
    if (zero != 0.f) {
        constexpr int STEP = EPI == TG_GATED ? 2 : 1;          // blocks of columns an output is made of
#pragma nounroll
        for (int i = 0; i < TMB; ++i) {
            uint64_t which = 0;                                // bit 16 * j + e
#pragma unroll
            for (int ii = 0; ii < TMB; ++ii)
#pragma unroll
                for (int j = 0; j < TNB; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        which |= static_cast<uint64_t>(ii == i && !__builtin_isfinite(acc[ii][j][e])) << (16 * (j / STEP) + e);
            static_assert(TNB * 16 <= 64, "a bit a number");
            for (; which; which &= which - 1) {
                const int bit = __builtin_ctzll(which), j = bit / 16, m = row_of(i, bit % 16);
                const int n = nt * (BN / STEP) + wn * (BN / WN / STEP) + 32 * j + (lane & 31);
                if (m >= M || n >= cols) continue;
                int row = m;
                if constexpr (GROUPED)
                    if (rows) row = rows[m];
                const float* xk = x + static_cast<size_t>(row) * K + kbeg;
                const float first = plain_dot(xk, w + static_cast<size_t>(n) * ldw + kbeg, kend - kbeg);
                float v;
                if constexpr (EPI == TG_GATED) v = act.value(first, plain_dot(xk, w + static_cast<size_t>(half + n) * ldw + kbeg, kend - kbeg));
                else v = act.plain(first);
                base[static_cast<size_t>(m) * cols + n] = v;
            }
        }
    }
}
