// Matrix products of many rows in float32: y[M, N] = x[M, K] . W[N, K]^T, where the time is the time of the matrix
// cores.
//
// gfx950 multiplies float32 operands at 157 TFLOP/s and bfloat16 operands at sixteen times that.  A float32 number is
// the sum of three bfloat16 numbers (24 bits of significand are three times 8):  x = xh + xm + xl, with xh rounded from x
// and xm from the rest; exactly, for numbers of 2^-110 and more (below that xl, whose last place is 2^-133, is rounded too).
// Of the nine products of two such sums the six largest are taken,
//     xl wh + xh wl + xm wm + xm wh + xh wm + xh wh,
// each product exact and added up in float32 by the matrix cores.  |xm| is at most 2^-8 |x| and |xl| 2^-17 |x|, so the three
// left out are at most 2^-24 of |x||w| and 2^-27.2 on average, no more than one float32 rounding.  (With xh cut off instead of
// rounded, which is up to 1.5 % faster, it was 2^-22 and 2^-25.2.)  Six bfloat16 instructions take 3/8 of the time of the float32 ones
// they replace.  What is left of the error is the sums': against 64 bits, relative to the root of the sum of the squared
// products, [512, 1024] with 1 / 16 / 256 numbers a row that are not zero 3.5e-8 / 1.6e-7 / 4.2e-7 where the library's float32
// product has 2.5e-8 / 7.4e-8 / 2.9e-7; sums of 700 to 8,192 numbers 0.6 to 0.9 times the library's.
//
// A workgroup owns BM rows of x and BN rows of W.  Both come from global memory as float32, BK at a time, wait in
// registers while the slab before them is multiplied, are taken apart there and written to LDS as three planes side by
// side; a row of a slab takes 3 * BK * 2 bytes and 16 more, so that the 16-byte reads of any eight neighbouring rows
// meet all banks.  LDS holds two slabs: one is read by the matrix instructions while the other is written.
// A matrix whose tiles would leave compute units idle is cut along K into shares, whose float32 sums a second kernel
// adds in their order.
//
// What bounds it is the matrix cores under load: a workgroup alone works at a rate that on 256 units were 1.82 PFLOP/s
// of bfloat16 products, all of them together reach 1.2 to 1.32 (the library's bfloat16 product of 8,192^3 1.41), as the
// clock falls.  Measured against the library's float32 product, recorded, every launch with another W (us): 512 rows on
// [16384, 2048] 259 : 172 (with SwiGLU 265 : 171), on [2048, 8192] 135 : 99, on [3072, 2048] 61 : 48, on [2048, 2048] 38 : 37;
// 1,999 rows on [16384, 2048] 930 : 607 (221 TFLOP/s).  Tiles: the larger the tile, the fewer reads of LDS and
// numbers taken apart a product; 256 x 256 runs at 220 TFLOP/s, 128 x 256 at 197, the smaller ones at 165 and fill the
// chip where there are few rows.
//
// An infinity less itself has no rest (nor has a number so large that it rounds to one): what it takes part in comes out
// of the matrix cores as NaN.  Numbers of the result
// that are not finite are therefore worked out again from the float32 operands (plain_dot), each by the lane that holds
// it, and are what a float32 product gives: infinities with their sign, NaN where there is no answer.  Finite results
// pay one multiplication; 1,999 rows on [16384, 2048] take 0.63 ms, 0.95 with an infinity in one row, 38 with one in every row.
#include "rope_store.h"
#include "row_stores.h"
#include "split_tile.h"

template <int BM, int BN, int WM, int WN, bool AHEAD, int EPI, bool GROUPED>
__global__ __launch_bounds__(WM * WN * WAVE) void split_gemm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                    float* __restrict__ out, int M, int N, int K, int kper,
                                                                    int mtiles, int ntiles, GatedUnit act, Groups groups) {
    __shared__ __attribute__((aligned(16))) char lds[SplitLds<BM, BN>::BYTES];
    const int t = tile_of_block(blockIdx.x, mtiles * ntiles);
    int m0 = (t % mtiles) * BM, ldw = K;
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
        M = end;                                        // the last place of this group and one
        w += e * groups.wstride;
        ldw = groups.ldw;
    }
    const int share = blockIdx.y;
    const int kbeg = share * kper, kend = min(K, kbeg + kper);
    split_tile<BM, BN, WM, WN, AHEAD, EPI, GROUPED>(x, w, out, M, N, K, m0, nt, share, kbeg, kend, ldw, groups.rows, act, SplitSlabs::in<BM, BN>(lds));
}

// out[i] = the sum of the shares' n numbers, in their order; V at a time (n is a multiple of V).
template <typename T, int V>
__global__ __launch_bounds__(256) void add_shares_kernel(const float* __restrict__ parts, T* __restrict__ out, size_t n, int shares,
                                                         GatedUnit act) {
    const size_t i = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * V;
    if (i >= n) return;
    float s[V], v[V];
    VecIO<float, V>::load(parts + i, s);
    for (int p = 1; p < shares; ++p) {
        VecIO<float, V>::load(parts + static_cast<size_t>(p) * n + i, v);
#pragma unroll
        for (int j = 0; j < V; ++j) s[j] += v[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) s[j] = act.plain(s[j]);
    VecIO<T, V>::store(out + i, s);
}

template <int BM, int BN, int WM, int WN, bool AHEAD>
static int launch_split(const float* x, const float* w, float* out, int M, int N, int K, int shares, int kper, int epi,
                        GatedUnit act, hipStream_t stream) {
    const int cols = epi == TG_GATED ? N / 2 : N, per = epi == TG_GATED ? BN / 2 : BN;
    const int mt = (M + BM - 1) / BM, nt = (cols + per - 1) / per;
    const dim3 grid(mt * nt, shares);
    if (epi == TG_GATED) {
        auto kernel = split_gemm_kernel<BM, BN, WM, WN, AHEAD, TG_GATED, false>;
        kernel<<<grid, WM * WN * WAVE, 0, stream>>>(x, w, out, M, N, K, K, mt, nt, act, Groups{});
    } else {
        auto kernel = split_gemm_kernel<BM, BN, WM, WN, AHEAD, TG_STORE, false>;
        kernel<<<grid, WM * WN * WAVE, 0, stream>>>(x, w, out, M, N, K, kper, mt, nt, act, Groups{});
    }
    return NI_LAUNCH_RESULT();
}

// tile: 0 = 64 x 256, 1 = 128 x 128, 2 = 128 x 256, 3 = 256 x 256 (rows of x, rows of W).  shares > 1: `out` takes the sums of every
// share of kper columns
NI_EXPORT int ni_split_gemm(const void* x, const void* w, void* out, int M, int N, int K, int tile, int shares, int kper,
                            int gated, int activation, int squared, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 4 || shares < 1 || (shares > 1 && (gated || squared || kper <= 0 || kper % 16 || static_cast<long>(shares - 1) * kper >= K)) || (gated && N % 2))
        return static_cast<int>(hipErrorInvalidValue);
    GatedUnit act = GatedUnit::of(activation);
    act.squared = squared != 0;
    const float *xf = static_cast<const float*>(x), *wf = static_cast<const float*>(w);
    float* of = static_cast<float*>(out);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (shares == 1) kper = K;
    switch (tile) {
        case 0: return launch_split<64, 256, 1, 4, true>(xf, wf, of, M, N, K, shares, kper, gated, act, s);
        case 1: return launch_split<128, 128, 2, 2, true>(xf, wf, of, M, N, K, shares, kper, gated, act, s);
        case 2: return launch_split<128, 256, 2, 4, true>(xf, wf, of, M, N, K, shares, kper, gated, act, s);
        case 3: return launch_split<256, 256, 2, 4, false>(xf, wf, of, M, N, K, shares, kper, gated, act, s);
        default: return static_cast<int>(hipErrorInvalidValue);
    }
}

// ---------------------------------------------------------------- bfloat16, 65 and more rows, the re-tiled matrix
// y[M, N] = x[M, K] . W[N, K]^T with W in the order in which the products of decode steps stream it ([tile of 16
// rows][piece of 64 columns][lane][32 bytes]): a lane's 32 bytes of a piece are two operands of
// v_mfma_f32_16x16x32_bf16, so W goes from memory into registers and never through LDS.  Only x does: LDS is what a
// product with both operands there runs out of (a 256 x 256 tile of such a kernel kept the matrix cores busy 52 % of
// the time with LDS at 46 % of its cycles and its barriers between).
//
// A workgroup is WN wavefronts side by side, each with TN tiles of W of its own and all BM rows of x; nothing of W is
// loaded twice in a workgroup.  x comes in slabs of 64 columns, three of them in LDS: one is multiplied, the next is
// complete, the third is written from registers that were loaded a slab earlier.  A half piece (32 columns) of W is
// loaded two halves before its turn, into the registers of the half before: three sets take turns.  Behind the
// products of each 16 rows of x their operand of the next half is read, so that reads of LDS run beside the products
// all the time and no operand is held twice.  W is the A operand: a lane then has four neighbouring columns of a row
// of y and stores them at once.
//
// Measured in recorded launches, every one with another W (us; the library's product, with SwiGLU its kernel too, o and down
// with the norm behind them : this): 512 rows on [16384, 2048] with SwiGLU 43.9 : 41.1, on [2048, 8192] 39.1 : 33.5, on
// [3072, 2048] 15.4 : 18.7, on [2048, 2048] 18.1 : 18.7; 128 rows 25.9 : 24.9, 25.6 : 19.6, 14.5 : 13.5, 15.5 : 11.9.  (With W
// at hand from the launch before 35.3, 25.5, 15.1 and 11.9 without the norm at 512 rows: the first operands of W come from
// memory a slab ahead, and that is what they wait for.)  Raising a wavefront's priority while it multiplies (s_setprio)
// was worth 39.6 -> 34.2.  Where there are tiles enough for it the library's 256 x 256 ones are ahead (1.27 PFLOP/s at 2,048
// rows against 1.06).
template <int N> struct Num { static constexpr int value = N; };

template <int WN, int TM, int TN, int MINW, int EPI, typename OUT>
__global__ __launch_bounds__(WN * WAVE, MINW) void tiled_gemm_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                    OUT* __restrict__ out, int M, int N, int K, int per,
                                                                    int mtiles, int ntiles, GatedUnit act, RopeStore rope) {
    constexpr int THREADS = WN * WAVE, BM = TM * 16, BNT = WN * TN;      // BNT: tiles of W a workgroup
    constexpr int ROWB = 128 + 16, SLAB = BM * ROWB;
    constexpr int CX = BM * 8 / THREADS;
    __shared__ __attribute__((aligned(16))) char lds[3 * SLAB];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    const int t = tile_of_block(blockIdx.x, mtiles * ntiles);
    const int m0 = (t % mtiles) * BM, nt = t / mtiles, share = blockIdx.y;
    const int pieces = K / 64, pbeg = share * per, pend = min(pieces, pbeg + per);
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(x), 0, M * K * 2, 0x00020000);
    // x: 16 bytes a thread and chunk, eight neighbouring threads a row
    int xsrc[CX], xdst[CX];
#pragma unroll
    for (int c = 0; c < CX; ++c) {
        const int i = tid + c * THREADS, r = i >> 3;
        xsrc[c] = min(m0 + r, M - 1) * K * 2 + (i & 7) * 16;
        xdst[c] = r * ROWB + (i & 7) * 16;
    }
    // W: tile, piece, lane, 32 bytes
    const int all = (N + 15) / 16;
    int wt[TN];                  // bytes from the start of W
    const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(w), 0, all * pieces * 2048, 0x00020000);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        int n;
        if constexpr (EPI == TG_GATED) {       // the first half of a wave's tiles are gate rows, the other half the up rows of the same outputs
            const int o = min(nt * (BNT / 2) + wave * (TN / 2) + j % (TN > 1 ? TN / 2 : 1), all / 2 - 1);
            n = (j / (TN > 1 ? TN / 2 : 1)) * (all / 2) + o;
        } else if constexpr (EPI == TG_ROPE) { // a wave's two tiles are sixteen dims of a head's first half and the ones half a head behind them
            static_assert(TN == 2, "a pair of tiles a wave");
            const int o = min(nt * (BNT / 2) + wave, all / 2 - 1), pairs = rope.hd / 32;
            n = o / pairs * 2 * pairs + o % pairs + j * pairs;
        } else {
            n = min(nt * BNT + wave * TN + j, all - 1);
        }
        wt[j] = (n * pieces * 64 + lane) * 32;
    }
    const int xoff = (lane & 15) * ROWB + (lane >> 4) * 32;
    u32x4_t xs[CX], wreg[3][TN];
    bf16x8_t xf[TM];
    floatx4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    int pos[TM], slot[TM];                                     // of the rows, with the rotation: long there when they are needed (512 rows on
                                                               // [3072, 2048] 16.6 -> 15.8 us, with the angles of all rows asked for together)
    if constexpr (EPI == TG_ROPE) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = min(m0 + i * 16 + (lane & 15), M - 1);
            pos[i] = rope.positions[m];
            slot[i] = rope.slots ? rope.slots[m] : -1;
        }
    }
    auto fetch = [&](int p) {
        const int at = min(p, pend - 1) * 128;
#pragma unroll
        for (int c = 0; c < CX; ++c) xs[c] = __builtin_amdgcn_raw_buffer_load_b128(xr, xsrc[c], at, 0);
    };
    auto put = [&](int buf) {
#pragma unroll
        for (int c = 0; c < CX; ++c) *reinterpret_cast<u32x4_t*>(lds + buf + xdst[c]) = xs[c];
    };
    auto weights = [&](u32x4_t (&r)[TN], int h) {        // half h of the share: piece pbeg + h / 2
        const int at = min(pbeg + (h >> 1), pend - 1) * 2048 + (h & 1) * 16;
#pragma unroll
        for (int j = 0; j < TN; ++j) r[j] = __builtin_amdgcn_raw_buffer_load_b128(wr, wt[j], at, 0);
    };
    auto read = [&](int i, int buf, int half) {
        xf[i] = *reinterpret_cast<const bf16x8_t*>(lds + buf + xoff + i * 16 * ROWB + half * 16);
    };
    fetch(pbeg);
    weights(wreg[0], 0);
    weights(wreg[1], 1);
    put(0);
    fetch(pbeg + 1);
    put(SLAB);
    fetch(pbeg + 2);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i) read(i, 0, 0);
    // half a piece: its operands are in registers; the next half's rows of x are read behind each row of tiles
    auto half = [&](const u32x4_t (&now)[TN], u32x4_t (&ahead)[TN], int h, int buf, int which) {
        weights(ahead, h + 2);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, now[j]), xf[i], acc[i][j], 0, 0, 0);
            read(i, buf, which);
        }
        __builtin_amdgcn_s_setprio(0);
    };
    // three pieces a turn: three slabs of x and three half pieces of W take turns
    auto piece = [&](auto B, int p) {
        constexpr int b = decltype(B)::value;                 // p % 3 counted from the share's first piece
        constexpr int h = 2 * b % 3;
        const int at = 2 * (p - pbeg);
        put((b + 2) % 3 * SLAB);
        fetch(p + 3);
        half(wreg[h], wreg[(h + 2) % 3], at, b * SLAB, 1);
        half(wreg[(h + 1) % 3], wreg[h], at + 1, (b + 1) % 3 * SLAB, 0);
        __syncthreads();
    };

    int p = pbeg;
    for (; p + 3 <= pend; p += 3) {
        piece(Num<0>{}, p);
        piece(Num<1>{}, p + 1);
        piece(Num<2>{}, p + 2);
    }
    if (p < pend) piece(Num<0>{}, p);
    if (p + 1 < pend) piece(Num<1>{}, p + 1);

    if constexpr (EPI == TG_ROPE) {
        const int o = nt * (BNT / 2) + wave, pairs = rope.hd / 32;
        if (o >= all / 2) return;
        const int head = o / pairs, d = o % pairs * 16 + (lane >> 4) * 4;
        RopeStore::Angles<4> t[TM];                            // of all rows, asked for together, behind one wait
#pragma unroll
        for (int i = 0; i < TM; ++i)
            if (rope.rotates(head)) t[i] = rope.angles<4>(pos[i], d);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = m0 + i * 16 + (lane & 15);
            if (m >= M) continue;
            const float a[4] = {acc[i][0][0], acc[i][0][1], acc[i][0][2], acc[i][0][3]}, b[4] = {acc[i][1][0], acc[i][1][1], acc[i][1][2], acc[i][1][3]};
            bf16_t* to = rope.place(m, slot[i], head);
            if (!to) continue;
            if (rope.rotates(head)) rope.turned<4>(to, d, a, b, t[i]);
            else rope.plain<4>(to, d, a, b);
        }
        return;
    }
    const int cols = EPI == TG_GATED ? N / 2 : N;
    OUT* base = out + static_cast<size_t>(share) * M * cols;
    constexpr int OT = EPI == TG_GATED && TN > 1 ? TN / 2 : TN, RUN = OT % 2 ? 1 : 2;      // RUN: stores that leave a row together
    struct __attribute__((aligned(4 * sizeof(OUT)))) Four { OUT v[4]; };
    const bool upper = RUN == 2 && (lane & 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + i * 16 + (RUN == 2 ? lane & 7 : lane & 15);
#pragma unroll
        for (int j = 0; j < OT; j += RUN) {
            const int n = (nt * (BNT * OT / TN) + wave * OT + j + upper) * 16 + (lane >> 4) * 4;
            Four o[RUN];
#pragma unroll
            for (int k = 0; k < RUN; ++k) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = EPI == TG_GATED ? act.rough(acc[i][j + k][e], acc[i][j + k + TN - OT][e]) : act.plain(acc[i][j + k][e]);
                store_packed<OUT, 4>(o[k].v, v);
            }
            if constexpr (RUN == 2) rows_together(o[0], o[1], upper);
            if (n >= cols) continue;
#pragma unroll
            for (int k = 0; k < RUN; ++k)
                if (m + 8 * k < M) *reinterpret_cast<Four*>(base + static_cast<size_t>(m + 8 * k) * cols + n) = o[k];
        }
    }
}

template <int WN, int TM, int TN, int MINW>
static int launch_tiled(const bf16_t* x, const bf16_t* w, void* out, int M, int N, int K, int shares, int per, int epi, int f32, GatedUnit act,
                        hipStream_t stream) {
    constexpr int BM = TM * 16, BNT = WN * TN, T = WN * WAVE;
    const int tiles = (N + 15) / 16, mt = (M + BM - 1) / BM;
    if (epi == TG_GATED) {
        if constexpr (TN > 1) {
            const int nt = (tiles / 2 + BNT / 2 - 1) / (BNT / 2);
            tiled_gemm_kernel<WN, TM, TN, MINW, TG_GATED, bf16_t><<<dim3(mt * nt), T, 0, stream>>>(x, w, static_cast<bf16_t*>(out), M, N, K, per, mt, nt, act, RopeStore{});
            return NI_LAUNCH_RESULT();
        }
        return static_cast<int>(hipErrorInvalidValue);
    }
    const int nt = (tiles + BNT - 1) / BNT;
    const dim3 grid(mt * nt, shares);
    if (f32) tiled_gemm_kernel<WN, TM, TN, MINW, TG_STORE, float><<<grid, T, 0, stream>>>(x, w, static_cast<float*>(out), M, N, K, per, mt, nt, act, RopeStore{});
    else tiled_gemm_kernel<WN, TM, TN, MINW, TG_STORE, bf16_t><<<grid, T, 0, stream>>>(x, w, static_cast<bf16_t*>(out), M, N, K, per, mt, nt, act, RopeStore{});
    return NI_LAUNCH_RESULT();
}

// tile: 0 = 128 x 256, 1 = 128 x 128, 2 = 64 x 128, 3 = 64 x 64 (rows of x, columns of y).  shares > 1: `out` takes float32 sums
// of every share of `per` pieces; f32: float32 results
NI_EXPORT int ni_tiled_gemm(const void* x, const void* w, void* out, int M, int N, int K, int tile, int shares, int per, int gated, int f32,
                            int activation, int squared, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 || N % 4 || shares < 1 || per < 1 || (shares > 1 && (!f32 || squared)) ||
        static_cast<long>(shares - 1) * per >= K / 64 || static_cast<long>(shares) * per < K / 64 || (gated && (N % 32 || shares > 1 || f32)) ||
        static_cast<long>(M) * K >= 1l << 30 || static_cast<long>(N + 15) * K >= 1l << 30)
        return static_cast<int>(hipErrorInvalidValue);
    GatedUnit act = GatedUnit::of(activation);
    act.squared = squared != 0;
    const bf16_t *xb = static_cast<const bf16_t*>(x), *wb = static_cast<const bf16_t*>(w);
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (tile) {
        case 0: return launch_tiled<8, 8, 2, 2>(xb, wb, out, M, N, K, shares, per, gated, f32, act, s);
        case 1: return launch_tiled<4, 8, 2, 2>(xb, wb, out, M, N, K, shares, per, gated, f32, act, s);
        case 2: return launch_tiled<4, 4, 2, 4>(xb, wb, out, M, N, K, shares, per, gated, f32, act, s);
        case 3: return launch_tiled<4, 4, 1, 4>(xb, wb, out, M, N, K, shares, per, gated, f32, act, s);
        default: return static_cast<int>(hipErrorInvalidValue);
    }
}

template <int WN, int TM, int MINW>
static int launch_tiled_rope(const bf16_t* x, const bf16_t* w, int M, int N, int K, const RopeStore& rope, hipStream_t stream) {
    constexpr int BM = TM * 16;
    const int mt = (M + BM - 1) / BM, nt = (N / 32 + WN - 1) / WN;
    tiled_gemm_kernel<WN, TM, 2, MINW, TG_ROPE, bf16_t><<<dim3(mt * nt), WN * WAVE, 0, stream>>>(x, w, static_cast<bf16_t*>(nullptr), M, N, K, K / 64, mt, nt, GatedUnit{}, rope);
    return NI_LAUNCH_RESULT();
}

// The product with the re-tiled stacked matrix [q; k; v] of (H + 2 KVH) heads of hd (whole pairs of 16): rotated queries to q, keys and values to
// the pools.  tile: 0, 1 or 2 of ni_tiled_gemm
NI_EXPORT int ni_tiled_qkv_rope(const void* x, const void* w, void* q, const void* positions, const void* cos_t, const void* sin_t, const void* slots, void* kpool,
                                void* vpool, int M, int K, int H, int KVH, int hd, int page_size, int tile, void* stream) {
    const long N = (H + 2l * KVH) * hd;
    if (M <= 0 || K <= 0 || K % 64 || H <= 0 || KVH <= 0 || hd <= 0 || hd % 32 || page_size <= 0 || static_cast<long>(M) * K >= 1l << 30 || (N + 15) * K >= 1l << 30 ||
        !q || !positions || !cos_t || !sin_t || (slots && (!kpool || !vpool)) ||
        (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kpool) | reinterpret_cast<uintptr_t>(vpool) |
         reinterpret_cast<uintptr_t>(cos_t) | reinterpret_cast<uintptr_t>(sin_t)) % 16)
        return static_cast<int>(hipErrorInvalidValue);
    const RopeStore rope{(const int32_t*)positions, (const float*)cos_t, (const float*)sin_t, (const int32_t*)slots, (bf16_t*)q, (bf16_t*)kpool, (bf16_t*)vpool,
                         H, KVH, hd, page_size};
    const bf16_t *xb = static_cast<const bf16_t*>(x), *wb = static_cast<const bf16_t*>(w);
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (tile) {
        case 0: return launch_tiled_rope<8, 8, 2>(xb, wb, M, static_cast<int>(N), K, rope, s);
        case 1: return launch_tiled_rope<4, 8, 2>(xb, wb, M, static_cast<int>(N), K, rope, s);
        case 2: return launch_tiled_rope<4, 4, 4>(xb, wb, M, static_cast<int>(N), K, rope, s);
        default: return static_cast<int>(hipErrorInvalidValue);
    }
}

// out[i] = (relu of, squared,) the sum of `shares` times n float32 numbers, in their order; four at a time where they and
// `out` start at whole vectors of four
NI_EXPORT int ni_add_shares(const void* parts, void* out, size_t n, int shares, int squared, int dtype, void* stream) {
    if (n == 0 || shares < 1) return static_cast<int>(hipErrorInvalidValue);
    GatedUnit act;
    act.squared = squared != 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool aligned = reinterpret_cast<uintptr_t>(parts) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % (dtype == 0 ? 16 : 8) == 0;
    const unsigned v = n % 4 == 0 && aligned ? 4 : 1, blocks = static_cast<unsigned>((n / v + 255) / 256);
    const float* pf = static_cast<const float*>(parts);
    if (dtype == 0) {
        if (v == 4) add_shares_kernel<float, 4><<<blocks, 256, 0, s>>>(pf, static_cast<float*>(out), n, shares, act);
        else add_shares_kernel<float, 1><<<blocks, 256, 0, s>>>(pf, static_cast<float*>(out), n, shares, act);
    } else {
        if (v == 4) add_shares_kernel<bf16_t, 4><<<blocks, 256, 0, s>>>(pf, static_cast<bf16_t*>(out), n, shares, act);
        else add_shares_kernel<bf16_t, 1><<<blocks, 256, 0, s>>>(pf, static_cast<bf16_t*>(out), n, shares, act);
    }
    return NI_LAUNCH_RESULT();
}

// ---------------------------------------------------------------- routed experts, every token with its own experts alone
// Every token has `top` entries (expert, weight).  The lists put the entries in the order of their experts, and an
// expert's entries in the order of the tokens: one workgroup an expert counts the entries of the experts before its own
// and then sets down its own, both in one order for all runs.  An entry that names no expert below E (an expert without
// matrices) stands in no list, its place is -1.
#define LIST_THREADS 1024
__global__ __launch_bounds__(LIST_THREADS) void expert_lists_kernel(const int32_t* __restrict__ chosen, const float* __restrict__ mix,
                                                                    int entries, int top, int E, int32_t* __restrict__ offsets,
                                                                    int32_t* __restrict__ rows, float* __restrict__ weights,
                                                                    int32_t* __restrict__ place) {
    constexpr int NW = LIST_THREADS / WAVE;
    __shared__ int counts[NW];
    const int e = blockIdx.x, lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    int before = 0;
    for (int i = threadIdx.x; i < entries; i += LIST_THREADS) {
        const int c = chosen[i];
        before += c >= 0 && c < e;
        if (e == 0 && (c < 0 || c >= E)) place[i] = -1;
    }
    __shared__ float scratch[16];
    int at = static_cast<int>(block_sum(static_cast<float>(before), scratch));      // whole numbers below 2^24
    if (threadIdx.x == 0) offsets[e] = at;
    for (int i0 = 0; i0 < entries; i0 += LIST_THREADS) {
        const int i = i0 + threadIdx.x;
        const bool mine = i < entries && chosen[i] == e;
        const unsigned long long votes = __ballot(mine);
        __syncthreads();
        if (lane == 0) counts[wave] = __popcll(votes);
        __syncthreads();
        int ahead = 0, all = 0;
#pragma unroll
        for (int v = 0; v < NW; ++v) {
            ahead += v < wave ? counts[v] : 0;
            all += counts[v];
        }
        if (mine) {
            const int p = at + ahead + __popcll(votes & ((1ull << lane) - 1));
            rows[p] = i / top;
            weights[p] = mix[i];
            place[i] = p;
        }
        at += all;
    }
    if (e == E - 1 && threadIdx.x == 0) offsets[E] = at;
}

// out[t, :] = the sum of what a token's entries gave, in the order of its entries
template <int V>
__global__ __launch_bounds__(256) void gather_entries_kernel(const float* __restrict__ y, const int32_t* __restrict__ place,
                                                             float* __restrict__ out, int d, int top) {
    const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * V;
    if (c >= d) return;
    float s[V], v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) s[j] = 0.f;
    for (int k = 0; k < top; ++k) {
        const int p = place[t * top + k];
        if (p < 0) continue;
        VecIO<float, V>::load(y + static_cast<size_t>(p) * d + c, v);
#pragma unroll
        for (int j = 0; j < V; ++j) s[j] += v[j];
    }
    VecIO<float, V>::store(out + static_cast<size_t>(t) * d + c, s);
}

NI_EXPORT int ni_expert_lists(const void* chosen, const void* mix, int T, int top, int E, void* offsets, void* rows, void* weights, void* place,
                              void* stream) {
    if (T <= 0 || top <= 0 || E <= 0 || static_cast<long>(T) * top >= (1 << 24)) return static_cast<int>(hipErrorInvalidValue);
    expert_lists_kernel<<<E, LIST_THREADS, 0, static_cast<hipStream_t>(stream)>>>((const int32_t*)chosen, (const float*)mix, T * top, top, E,
                                                                                  (int32_t*)offsets, (int32_t*)rows, (float*)weights, (int32_t*)place);
    return NI_LAUNCH_RESULT();
}

NI_EXPORT int ni_gather_entries(const void* y, const void* place, void* out, int T, int d, int top, void* stream) {
    if (T <= 0 || d <= 0 || top <= 0) return static_cast<int>(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool aligned = reinterpret_cast<uintptr_t>(y) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    if (d % 4 == 0 && aligned) gather_entries_kernel<4><<<dim3(T, (d / 4 + 255) / 256), 256, 0, s>>>((const float*)y, (const int32_t*)place, (float*)out, d, top);
    else gather_entries_kernel<1><<<dim3(T, (d + 255) / 256), 256, 0, s>>>((const float*)y, (const int32_t*)place, (float*)out, d, top);
    return NI_LAUNCH_RESULT();
}

template <int BM, int BN, int WM, int WN, bool AHEAD>
static int launch_grouped(const float* x, const float* w, float* out, int places, int N, int K, const Groups& groups, hipStream_t stream) {
    const int mt = places / BM + groups.count, nt = (N + BN - 1) / BN;      // at most: sum of ceil(rows / BM)
    split_gemm_kernel<BM, BN, WM, WN, AHEAD, TG_STORE, true><<<dim3(mt * nt, 1), WM * WN * WAVE, 0, stream>>>(x, w, out, places, N, K, K, mt, nt,
                                                                                                       GatedUnit{}, groups);
    return NI_LAUNCH_RESULT();
}

// out[p, n] = x[rows[p], :] . W[group of p][n, :] for every place p of the groups' lists
NI_EXPORT int ni_split_gemm_grouped(const void* x, const void* w, void* out, int places, int N, int K, const void* offsets, const void* rows,
                                    int count, size_t wstride, int ldw, int tile, void* stream) {
    if (places <= 0 || N <= 0 || K <= 0 || K % 4 || ldw < K || ldw % 4 || wstride % 4 || count <= 0) return static_cast<int>(hipErrorInvalidValue);
    const Groups g{static_cast<const int32_t*>(offsets), static_cast<const int32_t*>(rows), count, wstride, ldw};
    const float *xf = static_cast<const float*>(x), *wf = static_cast<const float*>(w);
    float* of = static_cast<float*>(out);
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (tile) {
        case 0: return launch_grouped<64, 256, 1, 4, true>(xf, wf, of, places, N, K, g, s);
        case 1: return launch_grouped<128, 128, 2, 2, true>(xf, wf, of, places, N, K, g, s);
        case 2: return launch_grouped<128, 256, 2, 4, true>(xf, wf, of, places, N, K, g, s);
        case 3: return launch_grouped<256, 256, 2, 4, false>(xf, wf, of, places, N, K, g, s);
        default: return static_cast<int>(hipErrorInvalidValue);
    }
}
