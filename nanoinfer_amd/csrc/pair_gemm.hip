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
// their way: a maximum over each wavefront in registers and four numbers in LDS (by atomics there it takes 3 us).  Measured, no such
// row : one in the first tile : one in every tile : all by tile_gemm.hip (us): 512 rows on [16384, 2048] with SwiGLU 110 : 191 : 206 : 178
// (looked at behind the main loop 107 : 249 : 290), on [2048, 8192] 69 : 111 : 121 : 103, on [2048, 2048] 25 : 37 : 37 : 38, 100 rows on
// [16384, 2048] 59 : 110 : 110 : 93, 2,000 rows there 355 : 478 : 760 : 610.
//
// Both operands come as halves: W once, when it is loaded, in the order of the lanes (pair_weight_kernel); x by a pass of its own
// (pair_rows_kernel, 3.5 to 8 us for 100 to 2,000 rows of 2,048).  A workgroup is four wavefronts side by side, one on each matrix core
// where the tile is largest, each with TN tiles of 32 rows of W and all 32 TM rows of x.  W goes from memory into registers three
// steps (of 16 columns) ahead of its turn and never through LDS: no two wavefronts share a row of it.  x comes in stages of 32
// columns through three slots of LDS; a stage's rows are loaded four stages ahead and written two ahead, and AHEAD the
// operands of a step are read during the step before (not where two workgroups share a unit and the registers do).
//
// Measured, recorded, every launch with another W, without the pass over x (us; six bfloat16 products : this): 512 rows on
// [16384, 2048] with SwiGLU 178 : 110, on [2048, 8192] 103 : 69, on [3072, 2048] 48 : 34, on [2048, 2048] 38 : 25; 2,000 rows on
// [16384, 2048] 610 : 355 (378 TFLOP/s); 100 rows on [16384, 2048] 93 : 59; 200 rows on [3072, 2048] 32 : 21.  What bounds it is the clock
// that the matrix cores hold: 256 workgroups of the largest tile take 0.68 us a step, eight 0.45 (of which the instructions are
// 0.32), and with operands of ones, which switch less, 256 take 0.56.  By counters, 2,048 rows on [16384, 2048]: 1.81 GHz, matrix cores busy
// 61 % of the cycles; 512 workgroups of the smallest tile: 2.30 GHz and 35 %.
#include "pair_rows.h"
#include "split_tile.h"

template <int N> struct Which { static constexpr int value = N; };

#define PAIR_TERMS 64           // products of big numbers that a result has at least

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

template <int TM, int TN, int SWM, int MINB, bool AHEAD, int EPI, bool GROUPED>
__global__ __launch_bounds__(256, MINB) void pair_gemm_kernel(const char* __restrict__ xp, const int2* __restrict__ xinfo, const char* __restrict__ wp,
                                                              const int2* __restrict__ winfo, const float* __restrict__ x,
                                                              const float* __restrict__ w, float* __restrict__ out, int M, int N, int K,
                                                              int kper, int wsteps, int mtiles, int ntiles, GatedUnit act, Groups groups,
                                                              PairGroups apart) {
    constexpr int BM = 32 * TM, BN = 128 * TN, R = 4;      // R: sixteens of columns of W in registers
    constexpr int ROWB = 128 + 16, SLAB = BM * ROWB, CX = BM * 8 / 256;
    constexpr int LDS = SplitLds<BM, BN>::BYTES > 3 * SLAB ? SplitLds<BM, BN>::BYTES : 3 * SLAB;
    __shared__ __attribute__((aligned(16))) char lds[LDS];
    __shared__ __attribute__((aligned(16))) int few_of[4], many_of[4];       // of every wavefront
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int t = tile_of_block(blockIdx.x, mtiles * ntiles);
    int m0 = (t % mtiles) * BM, ldw = K, rows = M, wtile = 0, wrow = 0, wstep = 0;
    const int nt = t / mtiles;
    if constexpr (GROUPED) {
        int tile = t % mtiles, e = 0, begin = 0, end = 0;
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
    const int sbeg = kbeg / 32, send = (kend + 31) / 32, rowb = ((K + 31) & ~31) * 4;

    auto row_at = [&](int m) {
        m = min(m, M - 1);
        if constexpr (GROUPED)
            if (groups.rows) m = groups.rows[m];
        return m;
    };
    // what the rows and columns of this tile were scaled by, and how many big numbers they have: waits in registers
    int2 mine_x = make_int2(0, INT_MAX), mine_w[(BN + 255) / 256];
    if (tid < BM) mine_x = xinfo[row_at(m0 + tid)];
#pragma unroll
    for (int c = 0; c < (BN + 255) / 256; ++c) {
        const int r = tid + c * 256;
        mine_w[c] = make_int2(0, 0);
        if (r < BN) {
            int n;
            if constexpr (EPI == TG_GATED) n = ((r >> 5) & 1) * half + min(nt * (BN / 2) + (r / 64) * 32 + (r & 31), half - 1);
            else n = min(nt * BN + r, N - 1);
            mine_w[c] = winfo[wrow + n];
        }
    }
    // x: 16 bytes a thread and chunk, eight neighbouring threads a row's 32 columns
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(xp), 0, INT_MAX, 0x00020000);
    int xsrc[CX], xdst[CX];
#pragma unroll
    for (int c = 0; c < CX; ++c) {
        const int i = tid + c * 256, r = i >> 3;
        xsrc[c] = row_at(m0 + r) * rowb + (i & 7) * 16;
        xdst[c] = r * ROWB + (i & 7) * 16;
    }
    // W: two planes of a lane's eight numbers for every tile of 32 rows and 16 columns
    int wsrc[TN];
    const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(wp), 0, INT_MAX, 0x00020000);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        int tile;
        if constexpr (EPI == TG_GATED) tile = (j & 1) * (half / 32) + min((nt * 4 + wave) * (TN / 2) + j / 2, half / 32 - 1);
        else tile = min((nt * 4 + wave) * TN + j, (N + 31) / 32 - 1);
        wsrc[j] = ((wtile + tile) * wsteps + wstep) * 2048;
    }
    struct Rows { u32x4_t v[CX]; };
    struct Cols { u32x4_t v[TN][2]; };
    struct Frags { f16x8_t v[2][TM]; };
    Rows xs[2];
    Cols wreg[R];
    Frags xf[AHEAD ? 2 : 1];
    floatx16_t acc[TM][TN], low[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = low[i][j][e] = 0.f;

    auto fetch = [&](Rows& r, int s) {
        const int at = min(s, send - 1) * 128;
#pragma unroll
        for (int c = 0; c < CX; ++c) r.v[c] = __builtin_amdgcn_raw_buffer_load_b128(xr, xsrc[c], at, 0);
    };
    auto put = [&](const Rows& r, int slot) {
#pragma unroll
        for (int c = 0; c < CX; ++c) *reinterpret_cast<u32x4_t*>(lds + slot + xdst[c]) = r.v[c];
    };
    auto weights = [&](Cols& r, int step) {               // sixteen columns: step counts from K's beginning
        const int at = min(step, 2 * send - 1) * 2048;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int p = 0; p < 2; ++p) r.v[j][p] = __builtin_amdgcn_raw_buffer_load_b128(wr, lane * 16 + p * 1024, wsrc[j] + at, 0);
    };
    const int xoff = (lane & 31) * ROWB + (lane >> 5) * 16;
    auto read = [&](Frags& f, int slot, int which) {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int i = 0; i < TM; ++i) f.v[p][i] = *reinterpret_cast<const f16x8_t*>(lds + slot + xoff + i * 32 * ROWB + which * 64 + p * 32);
    };
    auto multiply = [&](const Frags& a, const Cols& b) {
#pragma unroll
        for (int p = 0; p < 3; ++p) {                     // high by low, low by high, high by high
            constexpr int PA[3] = {0, 1, 0}, PB[3] = {1, 0, 0};
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    floatx16_t& to = p < 2 ? low[i][j] : acc[i][j];
                    to = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.v[PA[p]][i], __builtin_bit_cast(f16x8_t, b.v[j][PB[p]]), to, 0, 0, 0);
                }
        }
    };
    int at0 = 0, at1 = SLAB, at2 = 2 * SLAB;              // the slots of this stage, the next and the one behind it
    // 32 columns: their rows of x are in LDS, and the next 32; the ones behind are written, those behind them loaded
    auto stage = [&](auto B, int s) {
        constexpr int b = decltype(B)::value;
        put(xs[b], at2);
        fetch(xs[b], s + 4);
        weights(wreg[(2 * b + 3) % R], 2 * s + 3);
        if constexpr (AHEAD) read(xf[1], at0, 1);
        else read(xf[0], at0, 0);
        multiply(xf[0], wreg[2 * b]);
        weights(wreg[2 * b], 2 * s + 4);
        if constexpr (AHEAD) read(xf[0], at1, 0);
        else read(xf[0], at0, 1);
        multiply(xf[AHEAD ? 1 : 0], wreg[2 * b + 1]);
#pragma unroll
        for (int g = 0; g < 6 * TM * TN; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
        __syncthreads();
        const int first = at0;
        at0 = at1;
        at1 = at2;
        at2 = first;
    };
    // (in the order of the loop, so that what waits for the rows of x there does not wait for W)
    Rows first, second;
    fetch(first, sbeg);
    fetch(second, sbeg + 1);
    fetch(xs[0], sbeg + 2);
    fetch(xs[1], sbeg + 3);
#pragma unroll
    for (int r = 0; r < R - 1; ++r) weights(wreg[r], 2 * sbeg + r);
    // is there a result that these products may not be exact enough for
    int few = mine_x.y, many = mine_w[0].y;
#pragma unroll
    for (int c = 1; c < (BN + 255) / 256; ++c) many = max(many, mine_w[c].y);
    few = -wave_max(-few);
    many = wave_max(many);
    if (lane == 0) {
        few_of[wave] = few;
        many_of[wave] = many;
    }
    put(first, at0);
    put(second, at1);
    __syncthreads();
    const int4 f = *reinterpret_cast<const int4*>(few_of), m = *reinterpret_cast<const int4*>(many_of);
    few = __builtin_amdgcn_readfirstlane(min(min(f.x, f.y), min(f.z, f.w)));
    many = __builtin_amdgcn_readfirstlane(max(max(m.x, m.y), max(m.z, m.w)));
    if (few - PAIR_TERMS < many) {
        split_tile<BM, BN, SWM, 4 / SWM, true, EPI, GROUPED>(x, w, out, M, N, K, m0, nt, share, kbeg, kend, ldw, groups.rows, act, lds);
        return;
    }
    if constexpr (AHEAD) read(xf[0], at0, 0);
    int s = sbeg;
    for (; s + 2 <= send; s += 2) {
        stage(Which<0>{}, s);
        stage(Which<1>{}, s + 1);
    }
    if (s < send) stage(Which<0>{}, s);

    int* wexp = reinterpret_cast<int*>(lds);
    int* xexp = wexp + BN;
#pragma unroll
    for (int c = 0; c < (BN + 255) / 256; ++c)
        if (tid + c * 256 < BN) wexp[tid + c * 256] = mine_w[c].x;
    if (tid < BM) xexp[tid] = mine_x.x;
    __syncthreads();
    const int cols = EPI == TG_GATED ? half : N;
    float* base = out + static_cast<size_t>(share) * rows * cols;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int r = 32 * i + 8 * (e / 4) + 4 * (lane >> 5) + (e & 3), m = m0 + r;
            if (m >= M) continue;
            const int sx = xexp[r];
            auto value = [&](int j) { return ldexpf(fmaf(low[i][j][e], 1.f / 4096.f, acc[i][j][e]), -(sx + wexp[(wave * TN + j) * 32 + (lane & 31)])); };
            if constexpr (EPI == TG_GATED) {
#pragma unroll
                for (int j = 0; j < TN; j += 2) {
                    const int n = ((nt * 4 + wave) * (TN / 2) + j / 2) * 32 + (lane & 31);
                    if (n < cols) base[static_cast<size_t>(m) * cols + n] = act.value(value(j), value(j + 1));
                }
            } else {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int n = ((nt * 4 + wave) * TN + j) * 32 + (lane & 31);
                    if (n < cols) base[static_cast<size_t>(m) * cols + n] = act.plain(value(j));
                }
            }
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

template <int TM, int TN, int SWM, int MINB, bool AHEAD> static int launch_pair(const PairArgs& a) {
    constexpr int BM = 32 * TM, BN = 128 * TN;
    const int cols = a.gated ? a.N / 2 : a.N, per = a.gated ? BN / 2 : BN;
    const int mt = a.grouped ? a.M / BM + a.groups.count : (a.M + BM - 1) / BM, nt = (cols + per - 1) / per;
    const dim3 grid(mt * nt, a.shares);
#define PAIR_LAUNCH(EPI, GROUPED) pair_gemm_kernel<TM, TN, SWM, MINB, AHEAD, EPI, GROUPED><<<grid, 256, 0, a.stream>>>(a.xp, a.xinfo, a.wp, a.winfo, a.x, a.w, \
        a.out, a.M, a.N, a.K, a.kper, a.wsteps, mt, nt, a.act, a.groups, a.apart)
    if (a.grouped) PAIR_LAUNCH(TG_STORE, true);
    else if (a.gated) {
        if constexpr (TN % 2 == 0) PAIR_LAUNCH(TG_GATED, false);
        else return static_cast<int>(hipErrorInvalidValue);
    } else PAIR_LAUNCH(TG_STORE, false);
#undef PAIR_LAUNCH
    return NI_LAUNCH_RESULT();
}

static int launch_pair_tile(int tile, const PairArgs& a) {
    switch (tile) {
        case 0: return launch_pair<4, 2, 2, 1, true>(a);
        case 1: return launch_pair<2, 2, 1, 2, false>(a);
        case 2: return launch_pair<4, 1, 2, 2, false>(a);
        case 3: return launch_pair<2, 1, 2, 3, true>(a);
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
