// Products of many float32 rows, y[M, N] = x[M, K] . W[N, K]^T, by three products in half precision on the matrix cores.
//
// Brought to 2^14 .. 2^15 by a power of two that a whole row shares, a number is h + l / 4096 with halves h (rounded to nearest)
// and l (of the rest): two times 11 bits and the sign of l, so that what is left is at most one in the 24th bit, and exactly
// nothing for three numbers of four.  Of the four products of two such numbers three are taken,
//     y = 2^-(sx + sw) (sum xh wh + (sum xh wl + xl wh) / 4096),
// the two sums in accumulators of their own; xl wl is at most 2^-22 of a product and 2^-24.6 on average.  That is half the matrix
// instructions of the six bfloat16 products that do the same (tile_gemm.hip), and sums of half as many addends and fewer
// roundings: against 64 bits, relative to the root of the sum of the squared products, sums of 512 / 2,048 / 8,192 numbers
// 1.7e-7 / 3.0e-7 / 5.8e-7 where those have 3.4e-7 / 7.0e-7 / 1.4e-6 and the library's float32 product 4.1e-7 / 8.1e-7 / 1.6e-6.
//
// Where that is not so.  Halves have 30 binades: what is below 2^-12 of a scaled number's unit (2^-26 of its row's largest) loses
// bits, its error stays 2^-51 of the row's largest.  A number is big if it is at least 2^-12 and so more than 2^-13 of its
// row's largest.  Where a row of x has more big numbers than a row of W has others, at least one product of two big ones is in
// their sum, which makes sum |x||w| at least 2^-26 of the largest x times the largest w, and all that small numbers lose, 2 K 2^-51 of
// that at most, no more than K 2^-24 sum |x||w|: the bound of a float32 sum.  And with few addends the sum's roundings do not
// hide the halves': one product alone is off by 7e-8, 3.5e-8 in three parts.  So a tile in which some row of x has not at least
// PAIR_TERMS (64) more big numbers than some row of W has others is made by the six bfloat16 products (split_tile.h), by the
// same workgroup instead of its main loop; infinities and NaN count as no big number at all and end there too.  Normal
// deviates have one number in 2,900 that is not big, squared ReLU leaves half of them: neither gets there; a row of which one number
// is 30,000 times the rest does.  What is known of the rows is asked for before anything else and looked at while the first stages are on
// their way: a maximum over each wavefront in registers and a number of each in LDS (by atomics there it takes 3 us).  Measured, no such
// row : one in the first tile : one in every tile : all by tile_gemm.hip (us): 512 rows on [16384, 2048] with SwiGLU 84 : 164 : 181 : 173,
// on [2048, 8192] 53 : 97 : 103 : 91, on [2048, 2048] 16 : 39 : 40 : 31, 100 rows on [16384, 2048] 53 : 115 : 113 : 98, 2,000 rows
// there 343 : 591 : 715 : 628.
//
// Both operands come as halves: W once, when it is loaded, in the order of the lanes (pair_weight_kernel); x by a pass of its own
// (pair_rows_kernel, 3.5 to 8 us for 100 to 2,000 rows of 2,048) or by what makes x.  Both go from memory straight into LDS, without a
// register, in stages of 32 columns: 128 bytes of a row of x, whole lines (pieces of 64 bytes come at half the rate), their
// 16-byte pieces in another order for every second row, so that the reads meet no bank twice; W in the order that it is stored in,
// which the reads take as it is.  A ring holds three or four stages; of the one being multiplied the slots are asked for anew
// as soon as it is in registers, one barrier a stage.  A stage is three rounds of TM x TN products, low by high, high by
// low, high by high: what a round needs is read during the round before, so that no product waits for LDS.  (In the stages left over
// behind the loop, four of 64 in threes, the compiler waits for more loads than it has to.)  Where the registers are
// there, high by high has two sums that take the stages in turn: shorter sums have fewer roundings, so that a plan of half as many
// shares is no less exact (512 rows on [2048, 2048] in four shares 1.708e-7, in two with two sums 1.706e-7; kernels/tile.py keeps count).  Eight wavefronts, two on a matrix core, where the tile has the work for them:
// with four of them and 512 registers each the compiler keeps sums in accumulation registers and copies them (64 x 256: 110 us of
// 105).  The products are of 16 x 16, which draw less power than 32 x 32: the clock is 5 % higher.  Groups of PAIR_GROUP tiles of x share
// the tiles of W that they read from an L2; every group begins with another stage, so that what one die asks of memory first the next
// finds in the cache on the memory's side.
//
// Measured, recorded, every launch with another W, without the pass over x (us; six bfloat16 products : W in registers a stage of 16
// columns ahead, 32 x 32 products, four wavefronts : this): 512 rows on [16384, 2048] with SwiGLU 173 : 98 : 85, on [2048, 8192]
// 91 : 60 : 50, on [3072, 2048] 42 : 29 : 25, on [2048, 2048] 31 : 19 : 16; 1,500 rows on [2048, 8192] 150 : 125 (the second and this); 2,000 rows
// on [16384, 2048] 628 : 360 : 307 (437 TFLOP/s); 100 rows on [16384, 2048] 98 : 60 : 53; 200 rows on [3072, 2048] 28 : 20 : 17.  What
// bounds it is the clock that the matrix cores hold: by counters, 2,048 rows on [16384, 2048], they are busy 71 % of the cycles at
// 1.76 GHz (W in registers: 61 % at 1.81), 192 workgroups of the largest tile 47 % at 2.2 GHz; no bank conflicts.
#include "lds_load.h"
#include "pair_rows.h"
#include "split_tile.h"


#define PAIR_TERMS 64           // products of big numbers that a result has at least
#define PAIR_GROUP 4            // tiles of x side by side

template <int ROWS> struct Slot { char b[ROWS * 128]; };

// eight numbers of a row from k on, zeros behind its end; K is a multiple of four
__device__ __forceinline__ void load8(const float* __restrict__ row, int k, int K, float* v) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const float4 f = k + 4 * c < K ? *reinterpret_cast<const float4*>(row + k + 4 * c) : make_float4(0.f, 0.f, 0.f, 0.f);
        v[4 * c] = f.x; v[4 * c + 1] = f.y; v[4 * c + 2] = f.z; v[4 * c + 3] = f.w;
    }
}

__device__ __forceinline__ uint32_t top_bits(const float* v, uint32_t top) {
#pragma unroll
    for (int i = 0; i < 8; ++i) top = max(top, __float_as_uint(v[i]) & 0x7fffffffu);
    return top;
}

// A row's numbers, C chunks of eight a thread (C = 0: read again), and its thread's part of the row's largest bits, as pairs of halves; by a
// workgroup of 256.
template <int C>
__device__ __forceinline__ void row_to_pairs(float (&v)[C ? C : 1][8], uint32_t top, const float* __restrict__ row, int K, char* __restrict__ to,
                                             int2* __restrict__ info) {
    __shared__ uint32_t tops[4];
    __shared__ int bigs[4];
    const int kp = (K + 31) & ~31, tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), off, WAVE)));
    if (lane == 0) tops[wave] = top;
    __syncthreads();
    top = max(max(tops[0], tops[1]), max(tops[2], tops[3]));
    const int s = pair_scale(top);
    int big = 0;
    auto put = [&](float* u, int k) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            u[i] = ldexpf(u[i], s);
            big += fabsf(u[i]) >= PAIR_BIG;
        }
        uint4 h, l;
        pair_up(u, h, l);
        char* p = to + pair_place(k);
        *reinterpret_cast<uint4*>(p) = h;
        *reinterpret_cast<uint4*>(p + 32) = l;
    };
    if constexpr (C) {
#pragma unroll
        for (int c = 0; c < C; ++c)
            if ((tid + c * 256) * 8 < kp) put(v[c], (tid + c * 256) * 8);
    } else {
        for (int k = tid * 8; k < kp; k += 2048) {
            load8(row, k, K, v[0]);
            put(v[0], k);
        }
    }
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) big += __shfl_xor(big, off, WAVE);
    if (lane == 0) bigs[wave] = big;
    __syncthreads();
    if (tid == 0) {
        big = bigs[0] + bigs[1] + bigs[2] + bigs[3];
        *info = pair_row_info(s, top, big);
    }
}

// Rows of x: a workgroup a row, C chunks of eight numbers a thread in registers (C = 0: read twice).
template <int C>
__global__ __launch_bounds__(256) void pair_rows_kernel(const float* __restrict__ x, char* __restrict__ planes, int2* __restrict__ info, int K) {
    const int kp = (K + 31) & ~31, tid = threadIdx.x;
    const float* row = x + static_cast<size_t>(blockIdx.x) * K;
    float v[C ? C : 1][8];
    uint32_t top = 0;
    if constexpr (C) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int k = (tid + c * 256) * 8;
            load8(row, k, K, v[c]);
            top = top_bits(v[c], top);
        }
    } else {
        for (int k = tid * 8; k < kp; k += 2048) {
            load8(row, k, K, v[0]);
            top = top_bits(v[0], top);
        }
    }
    row_to_pairs<C>(v, top, row, K, planes + static_cast<size_t>(blockIdx.x) * kp * 4, info + blockIdx.x);
}

// Rows of x that are the merged key runs of an attention (what merge_splits_kernel of attention.hip makes of them, in the same order), and
// the same as pairs: a workgroup a token, C chunks of eight dims a thread.  part_o [T, H, runs, hd], part_ml [T, H, runs, 2] (maximum, sum).
template <int C>
__global__ __launch_bounds__(256) void merge_pair_rows_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml, float* __restrict__ x,
                                                              char* __restrict__ planes, int2* __restrict__ info, int H, int hd, int runs) {
    const int K = H * hd, kp = (K + 31) & ~31, t = blockIdx.x;
    float* row = x + static_cast<size_t>(t) * K;
    float v[C][8];
    uint32_t top = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int k = (threadIdx.x + c * 256) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[c][e] = 0.f;
        if (k < K) {
            const size_t p0 = (static_cast<size_t>(t) * H + k / hd) * runs;
            const int dim = k % hd;
            float M = -INFINITY, L = 0.f;
            for (int s = 0; s < runs; ++s) M = fmaxf(M, part_ml[(p0 + s) * 2]);
#pragma unroll 4
            for (int s = 0; s < runs; ++s) {
                const float f = expf(part_ml[(p0 + s) * 2] - M);
                float u[8];
                VecIO<float, 8>::load(part_o + (p0 + s) * hd + dim, u);
                L += part_ml[(p0 + s) * 2 + 1] * f;
#pragma unroll
                for (int e = 0; e < 8; ++e) v[c][e] += u[e] * f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] /= L;
            VecIO<float, 8>::store(row + k, v[c]);
        }
        top = top_bits(v[c], top);
    }
    row_to_pairs<C>(v, top, row, K, planes + static_cast<size_t>(t) * kp * 4, info + t);
}

// Rows of W: a workgroup 32 rows, in the order in which the product's wavefronts take them: [tile of 32 rows][16 columns]
// [plane][lane][16 bytes], lane = 32 * (which eight of the columns) + row.  info: scale, and how many numbers are not big.
#define PAIR_WEIGHT_WAVES 16
__global__ __launch_bounds__(PAIR_WEIGHT_WAVES * WAVE) void pair_weight_kernel(const float* __restrict__ w, char* __restrict__ planes, int2* __restrict__ info, int N, int K) {
    __shared__ uint32_t tops[32];
    __shared__ int bigs[32];
    const int kp = (K + 31) & ~31, tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE, n0 = blockIdx.x * 32;
    if (tid < 32) bigs[tid] = 0;
    for (int r = wave; r < 32; r += PAIR_WEIGHT_WAVES) {
        uint32_t top = 0;
        const float* row = w + static_cast<size_t>(n0 + r) * K;
        if (n0 + r < N)
            for (int k = lane * 8; k < K; k += WAVE * 8) {
                float v[8];
                load8(row, k, K, v);
                top = top_bits(v, top);
            }
#pragma unroll
        for (int off = WAVE / 2; off > 0; off >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), off, WAVE)));
        if (lane == 0) tops[r] = top;
    }
    __syncthreads();
    const int r = lane & 31;
    const uint32_t top = tops[r];
    const int s = pair_scale(top);
    const float* row = w + static_cast<size_t>(min(n0 + r, N - 1)) * K;
    char* to = planes + static_cast<size_t>(blockIdx.x) * kp * 128 + lane * 16;
    int big = 0;
    for (int t = wave; t < kp / 16; t += PAIR_WEIGHT_WAVES) {
        float v[8];
        load8(row, t * 16 + (lane >> 5) * 8, K, v);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = n0 + r < N ? ldexpf(v[i], s) : 0.f;
            big += fabsf(v[i]) >= PAIR_BIG;
        }
        uint4 h, l;
        pair_up(v, h, l);
        *reinterpret_cast<uint4*>(to + static_cast<size_t>(t) * 2048) = h;
        *reinterpret_cast<uint4*>(to + static_cast<size_t>(t) * 2048 + 1024) = l;
    }
    atomicAdd(&bigs[r], big);
    __syncthreads();
    if (tid < 32 && n0 + tid < N)
        info[n0 + tid] = make_int2(s, top == 0 ? 0 : top >= 0x7f800000u ? INT_MAX : K - bigs[tid]);
}

// The largest of a wavefront's numbers, in every lane.
__device__ __forceinline__ int wave_max(int v) {
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, false));       // of a row of sixteen lanes: row_ror:8, :4, :2, :1
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x124, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x122, 0xf, 0xf, false));
    v = max(v, __builtin_amdgcn_update_dpp(v, v, 0x121, 0xf, 0xf, false));
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = max(static_cast<int>(a[0]), static_cast<int>(a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return max(static_cast<int>(b[0]), static_cast<int>(b[1]));
}

// What tells the groups' rows of W apart, beside Groups.
struct PairGroups {
    int tiles;      // tiles of 32 rows of W from one group's to the next
    int steps;      // 16 columns from one group's to the next
};

template <int BM, int BN, int WM, int WN, int D, int EPI, bool GROUPED>
__global__ __launch_bounds__(WM * WN * WAVE, 2) void pair_gemm_kernel(const char* __restrict__ xp, const int2* __restrict__ xinfo, const char* __restrict__ wp,
                                                                     const int2* __restrict__ winfo, const float* __restrict__ x,
                                                                     const float* __restrict__ w, float* __restrict__ out, int M, int N, int K,
                                                                     int kper, int wsteps, int mtiles, int ntiles, GatedUnit act, Groups groups,
                                                                     PairGroups apart) {
    constexpr int NW = WM * WN, THREADS = NW * WAVE, TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int CX = BM / 8 / NW, CW = BN / 8 / NW, ALL = CX + CW;            // loads a wavefront and stage
    constexpr int SUMS = BM * BN <= 16384 ? 2 : 1;                                   // of high by high, stages in turn
    static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && BN <= THREADS && (EPI != TG_GATED || TN == 4) && TN % 2 == 0, "whole loads a wavefront");
    __shared__ __attribute__((aligned(1024))) Slot<BM> x0, x1, x2, x3;
    __shared__ __attribute__((aligned(1024))) Slot<BN> w0, w1, w2, w3;
    __shared__ __attribute__((aligned(16))) int few_of[NW], many_of[NW];     // of every wavefront
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wm = wave / WN, wn = wave % WN;
    const int t = tile_of_block(blockIdx.x, mtiles * ntiles);
    const int g = t / (PAIR_GROUP * ntiles), gm = min(PAIR_GROUP, mtiles - g * PAIR_GROUP), rem = t - g * PAIR_GROUP * ntiles;
    const int mt = g * PAIR_GROUP + rem % gm, nt = rem / gm;
    int m0 = mt * BM, ldw = K, rows = M, wtile = 0, wrow = 0, wstep = 0;
    if constexpr (GROUPED) {
        int tile = mt, e = 0, begin = 0, end = 0;
        for (; e < groups.count; ++e) {
            begin = groups.offsets[e];
            end = groups.offsets[e + 1];
            const int tiles = (end - begin + BM - 1) / BM;
            if (tile < tiles) break;
            tile -= tiles;
        }
        if (e == groups.count) return;
        m0 = begin + tile * BM;
        rows = M = end;
        w += e * groups.wstride;
        ldw = groups.ldw;
        wtile = e * apart.tiles;
        wrow = wtile * 32;
        wstep = e * apart.steps;
    }
    const int share = blockIdx.y;
    const int kbeg = share * kper, kend = min(K, kbeg + kper), half = N / 2;
    const int first = kbeg / 32, steps = (kend + 31) / 32 - first, rowb = ((K + 31) & ~31) * 4;
    const int turn = g * (steps / ((mtiles + PAIR_GROUP - 1) / PAIR_GROUP));         // the stage that this group begins with

    auto row_at = [&](int m) {
        m = min(m, M - 1);
        if constexpr (GROUPED)
            if (groups.rows) m = groups.rows[m];
        return m;
    };
    // tile of 32 rows of W at place q of the workgroup's: with SwiGLU a wavefront's two are gate rows and the up rows of the same outputs
    auto tile_at = [&](int q) {
        if constexpr (EPI == TG_GATED) return (q & 1) * (half / 32) + min(nt * (BN / 64) + q / 2, half / 32 - 1);
        else return min(nt * (BN / 32) + q, (N + 31) / 32 - 1);
    };
    // what the rows and columns of this tile were scaled by, and how many big numbers they have: waits in registers
    int2 mine_x = make_int2(0, INT_MAX), mine_w = make_int2(0, 0);
    if (tid < BM) mine_x = xinfo[row_at(m0 + tid)];
    if (tid < BN) mine_w = winfo[wrow + min(tile_at(tid / 32) * 32 + (tid & 31), N - 1)];
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(xp), 0, INT_MAX, 0x00020000);
    const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(wp), 0, INT_MAX, 0x00020000);
    int xsrc[CX], wsrc[CW];
#pragma unroll
    for (int c = 0; c < CX; ++c) {
        const int r = (wave + c * NW) * 8 + (lane >> 3);
        xsrc[c] = row_at(m0 + r) * rowb + ((lane & 7) ^ (r >> 1 & 7)) * 16;
    }
#pragma unroll
    for (int c = 0; c < CW; ++c) {
        const int q = wave + c * NW;                          // a quarter of a tile's 32 columns
        wsrc[c] = ((wtile + tile_at(q / 4)) * wsteps + wstep) * 2048 + q % 4 * 1024 + lane * 16;
    }
    floatx4_t acc[SUMS][TM][TN], low[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[0][i][j] = acc[SUMS - 1][i][j] = low[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    auto xslot = [&](auto I) -> Slot<BM>& {
        constexpr int i = decltype(I)::value % D;
        if constexpr (i == 0) return x0;
        else if constexpr (i == 1) return x1;
        else if constexpr (i == 2) return x2;
        else return x3;
    };
    auto wslot = [&](auto I) -> Slot<BN>& {
        constexpr int i = decltype(I)::value % D;
        if constexpr (i == 0) return w0;
        else if constexpr (i == 1) return w1;
        else if constexpr (i == 2) return w2;
        else return w3;
    };
    // loads FROM to TO of stage s, into slots I
    auto fetch = [&](auto I, int s, auto FROM, auto TO) {
        Slot<BM>& xs = xslot(I);
        Slot<BN>& ws = wslot(I);
        int at = min(s, steps - 1) + turn;
        at = first + at - (at >= steps ? steps : 0);
#pragma unroll
        for (int c = decltype(FROM)::value; c < decltype(TO)::value; ++c) {
            if (c < CX) load_to_lds(xr, xs.b + (wave + c * NW) * 1024, xsrc[c < CX ? c : 0], at * 128);
            else load_to_lds(wr, ws.b + (wave + (c - CX) * NW) * 1024, wsrc[c < CX ? 0 : c - CX], at * 4096);
        }
    };
    f16x8_t xh[TM], xl[TM], wl[TN], wh[2][TN];
    const int r = lane & 15, kg = lane >> 4;
    const int xo = ((wm * TM * 16 + r) * 128) + (((kg & 1) + (kg >> 1) * 4) ^ (r >> 1)) * 16;        // low halves two pieces on
    const int wo = wn * TN * 2048 + (kg >> 1) * 2048 + (kg & 1) * 512 + r * 16;                      // 1 KB on
    auto read_x = [&](f16x8_t (&f)[TM], auto I, int low_half) {
        const Slot<BM>& xs = xslot(I);
#pragma unroll
        for (int i = 0; i < TM; ++i) f[i] = *reinterpret_cast<const f16x8_t*>(xs.b + (low_half ? xo ^ 32 : xo) + i * 2048);
    };
    auto read_w = [&](f16x8_t (&f)[TN], auto I, int low_half) {
        const Slot<BN>& ws = wslot(I);
#pragma unroll
        for (int j = 0; j < TN; ++j) f[j] = *reinterpret_cast<const f16x8_t*>(ws.b + wo + low_half * 1024 + j / 2 * 4096 + j % 2 * 256);
    };
    auto multiply = [&](floatx4_t (&to)[TM][TN], const f16x8_t (&fx)[TM], const f16x8_t (&fw)[TN]) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fw[j], fx[i], to[i][j], 0, 0, 0);
    };
    // between the products: READS reads of operands, one behind each, and LOADS loads
    auto paced = [&](auto READS, auto LOADS) {
        constexpr int R = decltype(READS)::value, L = decltype(LOADS)::value, MF = TM * TN;
#pragma unroll
        for (int q = 0; q < MF; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (q < R) __builtin_amdgcn_sched_group_barrier(0x100, R > MF && q == 0 ? R - MF + 1 : 1, 0);
            if (q * L / MF != (q + 1) * L / MF) __builtin_amdgcn_sched_group_barrier(0x020, L > MF ? 2 : 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int L1 = (ALL + 2) / 3, L2 = L1 + (ALL + 1) / 3;
    // A stage: low by high, high by low, high by high.  What the first needs is in registers; during it the rest of the stage is read, then the
    // stage's slots are asked for anew and the first operands of the next stage read.
    auto stage = [&](auto I, int s) {
        constexpr int i = decltype(I)::value;
        read_x(xh, I, 0);
        read_w(wl, I, 1);
        fetch(Index<i + D - 1>{}, s + D - 1, Index<L2>{}, Index<ALL>{});
        multiply(low, xl, wh[i & 1]);
        paced(Index<TM + TN>{}, Index<ALL - L2>{});
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((D - 2) * ALL) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read_x(xl, Index<i + 1>{}, 1);
        fetch(I, s + D, Index<0>{}, Index<L1>{});
        multiply(low, xh, wl);
        paced(Index<TM>{}, Index<L1>{});
        read_w(wh[(i + 1) & 1], Index<i + 1>{}, 0);
        fetch(I, s + D, Index<L1>{}, Index<L2>{});
        multiply(acc[i % SUMS], xh, wh[i & 1]);
        paced(Index<TN>{}, Index<L2 - L1>{});
    };
    fetch(Index<0>{}, 0, Index<0>{}, Index<ALL>{});
    __builtin_amdgcn_sched_barrier(0);
    fetch(Index<1>{}, 1, Index<0>{}, Index<ALL>{});
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (D > 3) fetch(Index<2>{}, 2, Index<0>{}, Index<ALL>{});
    __builtin_amdgcn_sched_barrier(0);
    fetch(Index<D - 1>{}, D - 1, Index<0>{}, Index<L2>{});
    __builtin_amdgcn_sched_barrier(0);
    // is there a result that these products may not be exact enough for
    const int few_here = -wave_max(-mine_x.y), many_here = wave_max(mine_w.y);
    if (lane == 0) {
        few_of[wave] = few_here;
        many_of[wave] = many_here;
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((D - 2) * ALL + L2) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    int few = few_of[0], many = many_of[0];
#pragma unroll
    for (int v = 1; v < NW; ++v) {
        few = min(few, few_of[v]);
        many = max(many, many_of[v]);
    }
    few = __builtin_amdgcn_readfirstlane(few);
    many = __builtin_amdgcn_readfirstlane(many);
    if (few - PAIR_TERMS < many) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();                                      // nothing is on its way into the slots, which hold the slabs now
        constexpr int SNW = BM * 4 / WAVE < NW ? BM * 4 / WAVE : NW, SWN = BN / 64 < SNW ? BN / 64 : SNW, SWM = SNW / SWN;
        if (wave >= SNW) return;                              // (64 rows are work for four wavefronts; barriers wait for those that are left)
        split_tile<BM, BN, SWM, SWN, true, EPI, GROUPED>(x, w, out, M, N, K, m0, nt, share, kbeg, kend, ldw, groups.rows, act,
                                                         SplitSlabs{{x0.b, x1.b}, {w0.b, w1.b}});
        return;
    }
    read_x(xl, Index<0>{}, 1);
    read_w(wh[0], Index<0>{}, 0);
    constexpr int PERIOD = D % 2 ? 2 * D : D;
    int s = 0;
    for (; s + PERIOD <= steps; s += PERIOD) {
#define PAIR_STAGE(i) if constexpr (i < PERIOD) stage(Index<i>{}, s + i);
        PAIR_STAGE(0) PAIR_STAGE(1) PAIR_STAGE(2) PAIR_STAGE(3) PAIR_STAGE(4) PAIR_STAGE(5)
#undef PAIR_STAGE
    }
#define PAIR_STAGE(i) if constexpr (i + 1 < PERIOD) if (s + i < steps) stage(Index<i>{}, s + i);
    PAIR_STAGE(0) PAIR_STAGE(1) PAIR_STAGE(2) PAIR_STAGE(3) PAIR_STAGE(4)
#undef PAIR_STAGE
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    int *xexp = reinterpret_cast<int*>(x0.b), *wexp = reinterpret_cast<int*>(w0.b);
    if (tid < BM) xexp[tid] = mine_x.x;
    if (tid < BN) wexp[tid] = mine_w.x;
    __syncthreads();
    const int cols = EPI == TG_GATED ? half : N;
    float* base = out + static_cast<size_t>(share) * rows * cols;
    const bool vectors = cols % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    constexpr int OT = EPI == TG_GATED ? 2 : TN;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int mr = (wm * TM + i) * 16 + r, m = m0 + mr;
        if (m >= M) continue;
        const int sx = xexp[mr];
#pragma unroll
        for (int j = 0; j < OT; ++j) {
            const int n = EPI == TG_GATED ? (nt * (BN / 64) + wn) * 32 + j * 16 + kg * 4 : nt * BN + (wn * TN + j) * 16 + kg * 4;
            if (n >= cols) continue;
            auto value = [&](int block, int e) {
                const float high = SUMS == 1 ? acc[0][i][block][e] : acc[0][i][block][e] + acc[SUMS - 1][i][block][e];
                return ldexpf(fmaf(low[i][block][e], 1.f / 4096.f, high), -(sx + wexp[(wn * TN + block) * 16 + kg * 4 + e]));
            };
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (EPI == TG_GATED) v[e] = act.value(value(j, e), value(j + 2, e));
                else v[e] = act.plain(value(j, e));
            }
            float* to = base + static_cast<size_t>(m) * cols + n;
            if (vectors) VecIO<float, 4>::store(to, v);
            else
                for (int e = 0; e < 4 && n + e < cols; ++e) to[e] = v[e];
        }
    }
}

struct PairArgs {
    const char* xp;
    const int2* xinfo;
    const char* wp;
    const int2* winfo;
    const float *x, *w;
    float* out;
    int M, N, K, shares, kper, wsteps, gated;
    GatedUnit act;
    Groups groups;
    PairGroups apart;
    bool grouped;
    hipStream_t stream;
};

template <int BM, int BN, int WM, int WN, int D> static int launch_pair(const PairArgs& a) {
    const int cols = a.gated ? a.N / 2 : a.N, per = a.gated ? BN / 2 : BN;
    const int mt = a.grouped ? a.M / BM + a.groups.count : (a.M + BM - 1) / BM, nt = (cols + per - 1) / per;
    const dim3 grid(mt * nt, a.shares);
#define PAIR_LAUNCH(EPI, GROUPED) pair_gemm_kernel<BM, BN, WM, WN, D, EPI, GROUPED><<<grid, WM * WN * WAVE, 0, a.stream>>>(a.xp, a.xinfo, a.wp, a.winfo, a.x, a.w, \
        a.out, a.M, a.N, a.K, a.kper, a.wsteps, mt, nt, a.act, a.groups, a.apart)
    if (a.grouped) PAIR_LAUNCH(TG_STORE, true);
    else if (a.gated) {
        if constexpr (BN == 256) PAIR_LAUNCH(TG_GATED, false);
        else return static_cast<int>(hipErrorInvalidValue);
    } else PAIR_LAUNCH(TG_STORE, false);
#undef PAIR_LAUNCH
    return NI_LAUNCH_RESULT();
}

static int launch_pair_tile(int tile, const PairArgs& a) {
    switch (tile) {
        case 0: return launch_pair<128, 256, 2, 4, 3>(a);
        case 1: return launch_pair<64, 256, 2, 4, 3>(a);
        case 2: return launch_pair<128, 128, 4, 2, 4>(a);
        case 3: return launch_pair<64, 128, 2, 2, 3>(a);
        default: return static_cast<int>(hipErrorInvalidValue);
    }
}

NI_EXPORT int ni_pair_rows(const void* x, void* planes, void* info, int M, int K, void* stream) {
    if (M <= 0 || K <= 0 || K % 4) return static_cast<int>(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const float* xf = static_cast<const float*>(x);
    char* p = static_cast<char*>(planes);
    int2* i = static_cast<int2*>(info);
    if (K <= 2048) pair_rows_kernel<1><<<M, 256, 0, s>>>(xf, p, i, K);
    else if (K <= 4096) pair_rows_kernel<2><<<M, 256, 0, s>>>(xf, p, i, K);
    else if (K <= 8192) pair_rows_kernel<4><<<M, 256, 0, s>>>(xf, p, i, K);
    else pair_rows_kernel<0><<<M, 256, 0, s>>>(xf, p, i, K);
    return NI_LAUNCH_RESULT();
}

// hd a multiple of eight, H * hd at most 8,192; x [T, H * hd] takes the merged rows themselves
NI_EXPORT int ni_merge_pair_rows(const void* part_o, const void* part_ml, void* x, void* planes, void* info, int T, int H, int hd, int runs, void* stream) {
    if (T <= 0 || H <= 0 || hd <= 0 || hd % 8 || static_cast<long>(H) * hd > 8192 || runs < 1 || (reinterpret_cast<uintptr_t>(part_o) | reinterpret_cast<uintptr_t>(x)) % 16)
        return static_cast<int>(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const float *po = static_cast<const float*>(part_o), *ml = static_cast<const float*>(part_ml);
    float* xf = static_cast<float*>(x);
    char* p = static_cast<char*>(planes);
    int2* i = static_cast<int2*>(info);
    const int K = H * hd;
    if (K <= 2048) merge_pair_rows_kernel<1><<<T, 256, 0, s>>>(po, ml, xf, p, i, H, hd, runs);
    else if (K <= 4096) merge_pair_rows_kernel<2><<<T, 256, 0, s>>>(po, ml, xf, p, i, H, hd, runs);
    else merge_pair_rows_kernel<4><<<T, 256, 0, s>>>(po, ml, xf, p, i, H, hd, runs);
    return NI_LAUNCH_RESULT();
}

NI_EXPORT int ni_pair_weight(const void* w, void* planes, void* info, int N, int K, void* stream) {
    if (N <= 0 || K <= 0 || K % 4) return static_cast<int>(hipErrorInvalidValue);
    pair_weight_kernel<<<(N + 31) / 32, PAIR_WEIGHT_WAVES * WAVE, 0, static_cast<hipStream_t>(stream)>>>(static_cast<const float*>(w), static_cast<char*>(planes),
                                                                                  static_cast<int2*>(info), N, K);
    return NI_LAUNCH_RESULT();
}

// tile: 0 = 128 x 256, 1 = 64 x 256, 2 = 128 x 128, 3 = 64 x 128 (rows of x, rows of W).  xp, xinfo and wp, winfo: what ni_pair_rows and
// ni_pair_weight made of x and w.  shares > 1: `out` takes the sums of every share of kper columns.
NI_EXPORT int ni_pair_gemm(const void* xp, const void* xinfo, const void* wp, const void* winfo, const void* x, const void* w, void* out, int M, int N,
                           int K, int tile, int shares, int kper, int gated, int activation, int squared, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 4 || shares < 1 ||
        (shares > 1 && (gated || squared || kper <= 0 || kper % 32 || static_cast<long>(shares - 1) * kper >= K || static_cast<long>(shares) * kper < K)) ||
        (gated && N % 64))
        return static_cast<int>(hipErrorInvalidValue);
    PairArgs a{};
    a.xp = static_cast<const char*>(xp);
    a.xinfo = static_cast<const int2*>(xinfo);
    a.wp = static_cast<const char*>(wp);
    a.winfo = static_cast<const int2*>(winfo);
    a.x = static_cast<const float*>(x);
    a.w = static_cast<const float*>(w);
    a.out = static_cast<float*>(out);
    a.M = M;
    a.N = N;
    a.K = K;
    a.shares = shares;
    a.kper = shares == 1 ? K : kper;
    a.wsteps = (K + 31) / 32 * 2;
    a.gated = gated;
    a.act = GatedUnit::of(activation);
    a.act.squared = squared != 0;
    a.stream = static_cast<hipStream_t>(stream);
    return launch_pair_tile(tile, a);
}

// out[p, n] = x[rows[p], :] . W[group of p][n, :] for every place p of the groups' lists; the groups' rows of W stand one behind the
// other (down = 0: `per` = N of them each) or side by side (down = 1: K columns each).  wk: columns of the whole matrix W
NI_EXPORT int ni_pair_gemm_grouped(const void* xp, const void* xinfo, const void* wp, const void* winfo, const void* x, const void* w, void* out,
                                   int places, int N, int K, const void* offsets, const void* rows, int count, int down, int tile, void* stream) {
    if (places <= 0 || N <= 0 || K <= 0 || K % 32 || count <= 0 || (!down && N % 32)) return static_cast<int>(hipErrorInvalidValue);
    PairArgs a{};
    a.xp = static_cast<const char*>(xp);
    a.xinfo = static_cast<const int2*>(xinfo);
    a.wp = static_cast<const char*>(wp);
    a.winfo = static_cast<const int2*>(winfo);
    a.x = static_cast<const float*>(x);
    a.w = static_cast<const float*>(w);
    a.out = static_cast<float*>(out);
    a.M = places;
    a.N = N;
    a.K = K;
    a.shares = 1;
    a.kper = K;
    a.grouped = true;
    const size_t wide = down ? static_cast<size_t>(K) * count : K;
    a.wsteps = static_cast<int>(wide / 16);
    a.groups = Groups{static_cast<const int32_t*>(offsets), static_cast<const int32_t*>(rows), count, down ? static_cast<size_t>(K) : static_cast<size_t>(N) * K,
                      static_cast<int>(wide)};
    a.apart = PairGroups{down ? 0 : N / 32, down ? K / 16 : 0};
    a.stream = static_cast<hipStream_t>(stream);
    return launch_pair_tile(tile, a);
}
