// Products of many bfloat16 rows, y[M, N] = x[M, K] . W[N, K]^T, both operands as stored, with SwiGLU or squared ReLU in the epilogue.
//
// x and W go from memory straight into LDS (sixteen bytes a lane) and from there into the matrix cores' registers; no operand waits in
// registers for LDS.  A stage is 64 columns of K: 128 bytes of a row, one line.  (With 32 columns a stage, half a line a row, a compute
// unit takes in 69 GB/s whatever the source, with whole lines 137: a 256 x 256 tile 131 -> 116 us.)  Rows lie in LDS without gaps, as
// such a load leaves them; which of a row's eight pieces of sixteen bytes stands where is turned round by the row's number when it is
// asked for (wide_swizzle), so that the sixteen lanes that LDS serves at once meet no bank twice (counted: none).
//
// LDS is rings of stages, DX of x and DW of W.  While a half of a stage (32 columns) is multiplied the operands of the next half are
// read, in a second set of registers; when a wavefront has read a stage it waits until its own loads of the next one have
// landed, meets the others, and only then are the stage's places asked for anew: one barrier a stage, and loads have DX - 1 stages
// and more to arrive.  x goes first, W a stage further ahead where LDS has room for it (two stages of each, 256 x 256 tiles: 5 % slower): W
// comes from memory, x mostly from the caches.  Every ring slot is an array of its own, by which the compiler knows that a read in the loop
// does not wait for loads into the others.  (In the stages left over behind it, where ways join, it waits for more than it has to: two of 32 stages on
// 256 x 256 tiles with 2,048 columns.)
//
// The rows of x are taken in groups of WIDE_GROUP tiles, whose workgroups run on one die and share the lines of W in its L2; every
// group begins at another stage of K, so that of two dies that need the same W one asks memory for the half that the other finds in
// the memory-side cache: a unit has some 48 KB of lines on their way, 60 GB/s from memory and 115 from that cache
// ([2048, 8192] at 1,536 rows 66 -> 55 us, [3072, 2048] at 1,999 30.6 -> 27.5; groups of eight tiles 62, of two as fast, but 21 us
// for [2048, 2048] at 1,999 rows instead of 18).
//
// W is the first operand, and MFMA row 4 g + e of a block stands for row 16 g + 4 (block mod 4) + e of the tile's 64: a lane then holds sixteen
// neighbouring columns of a row of y and stores whole vectors.  With SwiGLU a wavefront's blocks are half gate rows, half the up rows of
// the same outputs.  Eight wavefronts, two a matrix core: given the whole register file (four wavefronts) the compiler moves
// accumulators between its halves.  v_mfma_f32_16x16x32 instead of 32x32x16: 114 -> 107 us for [16384, 2048] at 1,999 rows, as the clock holds
// 1.92 instead of 1.82 GHz.
//
// Measured (us, the library's product and the SwiGLU kernel : this; kernels/tile.py has more): [16384, 2048] with SwiGLU at 512 / 1,024 / 1,999 / 4,096 rows
// 44 : 36, 68 : 58, 121 : 111, 239 : 211; [2048, 8192] at 1,999 70 : 62.  Of [16384, 2048] at 1,999 rows the library's product alone takes 105: what is ahead is the
// epilogue.  17 to 64 rows on a head of [128256, 2048], where W streams from memory once and 64 rows of x from the caches for every tile: tiles of 64 x 128, two a
// unit so that one's start and stores go beside the other's stages, 115.8 us at 32 rows and 124.1 at 64 (the library's 120.9 and 130.6; tiles of 64 x 256 119.5
// and 129.6); on rows of 2,304 to 3,584 elements 64 x 256 ([128256, 3072] 150.7 and 160.7, the library's 167.7 and 184.9).
// Its loop runs at 1.42 PFLOP/s (kernels/tile.py: 1.509 us for 64 columns with all units at work), the launch at 1.2, and 1.1 to 1.2 inside a prompt: two rounds of
// one workgroup a unit, whose first loads and stores nothing covers.  In the loop it is the clock: alone, matrix cores busy 64 % of the time at 1.9 GHz
// (the library's 65 % at 1.96; with operands of ones, which switch less, 2.3 GHz and 88 us; without its loads the same kernel takes 103), in a prompt of 2,048
// tokens 57 % at 1.99.  A prompt of 1,999 tokens of the 1B shape 5,170 -> 4,630 us.
#include "lds_load.h"
#include "rope_store.h"
#include "row_norm.h"
#include "row_stores.h"
#include "split_tile.h"

// Which piece of sixteen bytes of row r stands where the row's piece 0 would.
__device__ __forceinline__ int wide_swizzle(int r) { return (r & 2) << 1 | ((r >> 4 ^ r >> 5) & 1) << 1 | (r >> 4 & 1); }

#define WIDE_GROUP 4            // tiles of x side by side

template <int ROWS> struct WideSlot { char b[ROWS * 128]; };

template <int BM, int BN, int WM, int WN, int DX, int DW, int EPI, typename OUT, bool NORMED>
__global__ __launch_bounds__(WM * WN * WAVE, 2) void wide_gemm_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                            OUT* __restrict__ out, int M, int N, int K, int mtiles,
                                                                            int ntiles, GatedUnit act, RopeStore rope, StreamStore stream, RowNorm norm) {
    constexpr int NW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int CX = BM / 8 / NW, CW = BN / 8 / NW, ALL = CX + CW;            // loads a wavefront and stage
    static_assert((TM % 4 == 0 || TM == 2) && TN % 4 == 0 && BM % (8 * NW) == 0 && BN % (8 * NW) == 0, "whole groups of 64 rows, whole loads a wavefront");
    static_assert(DX >= 2 && DW >= DX && DW <= 5, "slots");
    __shared__ __attribute__((aligned(1024))) WideSlot<BM> x0, x1, x2, x3, x4;
    __shared__ __attribute__((aligned(1024))) WideSlot<BN> w0, w1, w2, w3, w4;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int wm = wave / WN, wn = wave % WN;
    const int t = tile_of_block(blockIdx.x, mtiles * ntiles);
    const int g = t / (WIDE_GROUP * ntiles), gm = min(WIDE_GROUP, mtiles - g * WIDE_GROUP), rem = t - g * WIDE_GROUP * ntiles;
    const int m0 = (g * WIDE_GROUP + rem % gm) * BM, nt = rem / gm;
    const int steps = K / 64;
    const int turn = g * (steps / ((mtiles + WIDE_GROUP - 1) / WIDE_GROUP));          // the stage that this group begins with
    const int half = N / 2;
    // where the columns of block j and lane group q of a wavefront start: GB blocks stand side by side in a lane's run, as many as one store
    // takes, so that it leaves no holes between the lanes of a row (2,045 rows on [3072, 2048] to float32 33.7 us in runs of four blocks, 29.7 so, 29.0
    // with eight lanes of a row together: rows_together)
    constexpr int GB = EPI == TG_ROPE ? 2 : 4 / sizeof(OUT);
    auto column = [](int j, int q) { return j / GB * GB * 16 + q * GB * 4 + j % GB * 4; };
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(x), 0, M * K * 2, 0x00020000);
    const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(w), 0, N * K * 2, 0x00020000);
    int xsrc[CX], wsrc[CW];
#pragma unroll
    for (int c = 0; c < CX; ++c) {
        const int r = (wave + c * NW) * 8 + (lane >> 3);
        xsrc[c] = min(m0 + r, M - 1) * K * 2 + ((lane & 7) ^ wide_swizzle(r)) * 16;
    }
#pragma unroll
    for (int c = 0; c < CW; ++c) {
        const int r = (wave + c * NW) * 8 + (lane >> 3);
        int n;
        if constexpr (EPI == TG_GATED) {       // gate rows are the first half of a wavefront's blocks, the up rows of the same outputs the other
            const int wv = r / (TN * 16), b = r / 64 % (TN / 4) * 4 + (r >> 2 & 3);
            n = b / (TN / 2) * half + min(nt * (BN / 2) + wv * (TN * 8) + column(b % (TN / 2), r >> 4 & 3) + (r & 3), half - 1);
        } else if constexpr (EPI == TG_ROPE) { // 64 columns are 32 neighbouring dims of a head's first half and the 32 half a head behind them
            const int set = min(nt * (BN / 64) + r / 64, N / 64 - 1), sets = rope.hd / 64, b = r >> 2 & 3;
            n = set / sets * rope.hd + b / 2 * (rope.hd / 2) + set % sets * 32 + column(b % 2, r >> 4 & 3) + (r & 3);
        } else {
            n = min(nt * BN + (r & ~63) + column(r >> 2 & 3, r >> 4 & 3) + (r & 3), N - 1);
        }
        wsrc[c] = n * K * 2 + ((lane & 7) ^ wide_swizzle(r)) * 16;
    }
    floatx4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    auto xslot = [&](auto I) -> WideSlot<BM>& {
        constexpr int i = decltype(I)::value % DX;
        if constexpr (i == 0) return x0;
        else if constexpr (i == 1) return x1;
        else if constexpr (i == 2) return x2;
        else if constexpr (i == 3) return x3;
        else return x4;
    };
    auto wslot = [&](auto I) -> WideSlot<BN>& {
        constexpr int i = decltype(I)::value % DW;
        if constexpr (i == 0) return w0;
        else if constexpr (i == 1) return w1;
        else if constexpr (i == 2) return w2;
        else if constexpr (i == 3) return w3;
        else return w4;
    };
    // loads FROM to TO of the batch that may go out when stage s (in slots I) has been read: x of stage s + DX, then W of stage s + DW
    auto fetch = [&](auto I, int s, auto FROM, auto TO) {
        WideSlot<BM>& xs = xslot(I);
        WideSlot<BN>& ws = wslot(I);
        auto columns = [&](int s) {
            const int at = min(s, steps - 1) + turn;
            return (at - (at >= steps ? steps : 0)) * 128;
        };
        const int xat = columns(s + DX), wat = columns(s + DW);
#pragma unroll
        for (int c = decltype(FROM)::value; c < decltype(TO)::value; ++c) {
            if (c < CX) load_to_lds(xr, xs.b + (wave + c * NW) * 1024, xsrc[c < CX ? c : 0], xat);
            else load_to_lds(wr, ws.b + (wave + (c - CX) * NW) * 1024, wsrc[c < CX ? 0 : c - CX], wat);
        }
    };
    struct Frags { bf16x8_t x[TM], w[TN]; };
    Frags f[2];
    const int row = (lane >> 2 & 3) * 16 + (lane & 3);
    const int xblock = wm * TM;                                // this wavefront's first sixteen rows
    int xo[2], wo[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int at = ((k * 4 + (lane >> 4)) ^ wide_swizzle(row)) * 16;
        xo[k] = (xblock / 4 * 64 + xblock % 4 * 4 + row) * 128 + at;
        wo[k] = (wn * TN * 16 + row) * 128 + at;
    }
    auto read = [&](Frags& fr, auto I, int k) {
        const WideSlot<BM>& xs = xslot(I);
        const WideSlot<BN>& ws = wslot(I);
#pragma unroll
        for (int i = 0; i < TM; ++i) fr.x[i] = *reinterpret_cast<const bf16x8_t*>(xs.b + xo[k] + (i / 4) * 8192 + (i % 4) * 512);
#pragma unroll
        for (int j = 0; j < TN; ++j) fr.w[j] = *reinterpret_cast<const bf16x8_t*>(ws.b + wo[k] + (j / 4) * 8192 + (j % 4) * 512);
    };
    auto multiply = [&](const Frags& fr) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fr.w[j], fr.x[i], acc[i][j], 0, 0, 0);
    };
    // between the products: the reads of the next operands, one every second, and LOADS loads
    auto paced = [&](auto LOADS) {
        constexpr int L = decltype(LOADS)::value;
#pragma unroll
        for (int q = 0; q < TM * TN; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (TM * TN < 2 * (TM + TN) || (q % 2 == 0 && q / 2 < TM + TN)) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (q * L / (TM * TN) != (q + 1) * L / (TM * TN)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // loads that may still be on their way when the next stage is read: all that were asked for after its last one
    constexpr int WAITX = CW + (DX - 2) * ALL, WAITW = (DW - 2) * ALL, WAIT = WAITX < WAITW ? WAITX : WAITW;
    constexpr int FIRST = (ALL + 1) / 2;
    // (inside a half of a stage the compiler may order loads as it likes, and before the first stage inside a batch)
    static_assert(DX == DW || FIRST == CX, "batches are counted whole, or x in the first half of a stage and W in the second");
    auto stage = [&](auto I, int s) {
        constexpr int i = decltype(I)::value;
        read(f[1], I, 1);
        fetch(Index<i + DX * DW - 1>{}, s - 1, Index<FIRST>{}, Index<ALL>{});
        multiply(f[0]);
        paced(Index<ALL - FIRST>{});
        // this wavefront has read the stage, and its loads of the next one have landed; behind the barrier, every wavefront's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(WAIT) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        read(f[0], Index<i + 1>{}, 0);
        fetch(I, s, Index<0>{}, Index<FIRST>{});
        multiply(f[1]);
        paced(Index<FIRST>{});
    };
    // what stages before the first one would have asked for, in their order
    auto ahead = [&](auto B) {
        constexpr int b = decltype(B)::value;                  // stages before the first
        constexpr int last = b == 1 ? FIRST : ALL;
        if constexpr (b <= DX) fetch(Index<DX * DW - b>{}, -b, Index<0>{}, Index<(last < CX ? last : CX)>{});
        if constexpr (DX != DW) __builtin_amdgcn_sched_barrier(0);     // (x and W of different stages: the wait below counts x's first)
        if constexpr (b <= DW) fetch(Index<DX * DW - b>{}, -b, Index<CX>{}, Index<(last < CX ? CX : last)>{});
        __builtin_amdgcn_sched_barrier(0);
    };
    RowSquares<BM, NW * WAVE> squares;
    if constexpr (NORMED) squares.ask(norm, m0, M, tid);
    ahead(Index<5>{});
    ahead(Index<4>{});
    ahead(Index<3>{});
    ahead(Index<2>{});
    ahead(Index<1>{});
    const float factor = NORMED ? squares.factor(norm, K) : 1.f;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WAIT + FIRST) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(f[0], Index<0>{}, 0);
    constexpr int PERIOD = DX == DW ? DX : DX * DW;
    int s = 0;
    for (; s + PERIOD <= steps; s += PERIOD) {
#define WIDE_STAGE(i) if constexpr (i < PERIOD) stage(Index<i>{}, s + i);
        WIDE_STAGE(0) WIDE_STAGE(1) WIDE_STAGE(2) WIDE_STAGE(3) WIDE_STAGE(4) WIDE_STAGE(5)
#undef WIDE_STAGE
    }
#define WIDE_STAGE(i) if constexpr (i + 1 < PERIOD) if (s + i < steps) stage(Index<i>{}, s + i);
    WIDE_STAGE(0) WIDE_STAGE(1) WIDE_STAGE(2) WIDE_STAGE(3) WIDE_STAGE(4)
#undef WIDE_STAGE
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");           // (loads of stages behind the last: they land before the wavefront ends)

    auto factor_of = [&](int i) {                              // of this lane's row of block i
        if constexpr (NORMED) return reinterpret_cast<const float*>(x0.b)[(xblock + i) / 4 * 64 + (xblock + i) % 4 * 4 + row];
        else return 1.f;
    };
    if constexpr (NORMED) {
        __syncthreads();                                       // nobody reads or fills the ring any more
        constexpr int EACH = NW * WAVE / BM;
        if (tid % EACH == 0) reinterpret_cast<float*>(x0.b)[tid / EACH] = factor;
        __syncthreads();
    }
    if constexpr (EPI == TG_STREAM) {
        static_assert(TN == 4, "64 columns a wavefront, a part of a row's sum of squares");
        // lane by lane what rows_together leaves it: four columns of blocks j and j + 1 of a row and of the one 32 further on
        const int side = lane & 8 ? 16 : 0;
        auto stream_n = [&](int j) { return nt * BN + (wn * TN + j) * 16 + side + (lane >> 4) * 4; };
        float4 weight[TN / 2];
#pragma unroll
        for (int j = 0; j < TN; j += 2)
            weight[j / 2] = stream.next ? *reinterpret_cast<const float4*>(stream.weight + min(stream_n(j), N - 4)) : make_float4(0.f, 0.f, 0.f, 0.f);
        const bool here = nt * BN + wn * 64 < N;              // N is whole sets of 64
        auto row_at = [&](int i, int k) { return m0 + (xblock + i) / 4 * 64 + (xblock + i) % 4 * 4 + (row & 31) + 32 * k; };
        // what the stream holds, GROUP blocks of rows at a time: no load behind a store that it waits for
        constexpr int GROUP = TM < 4 ? TM : 4;
        float4 before[GROUP][TN];
        auto load = [&](int i0) {
#pragma unroll
            for (int i = 0; i < GROUP; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    before[i][j] = *reinterpret_cast<const float4*>(stream.h + static_cast<size_t>(min(row_at(i0 + i, j & 1), M - 1)) * N + min(stream_n(j & ~1), N - 4));
        };
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if (i % GROUP == 0) load(i);
            float sum[2] = {0.f, 0.f};
            uint2 next[2][TN / 2];
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                float4 o[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) o[k] = make_float4(acc[i][j + k][0], acc[i][j + k][1], acc[i][j + k][2], acc[i][j + k][3]);
                rows_together(o[0], o[1], side != 0);
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const float4 b = before[i % GROUP][j + k], w4 = weight[j / 2];
                    const float4 v = make_float4(b.x + o[k].x, b.y + o[k].y, b.z + o[k].z, b.w + o[k].w);
                    sum[k] += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
                    if (here && row_at(i, k) < M) *reinterpret_cast<float4*>(stream.h + static_cast<size_t>(row_at(i, k)) * N + stream_n(j)) = v;
                    next[k][j / 2] = make_uint2(pack_bf16x2(v.x * w4.x, v.y * w4.y), pack_bf16x2(v.z * w4.z, v.w * w4.w));
                }
            }
            if (stream.next) {
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    // lane groups 0 and 2 give their four columns of the second pair of blocks for the next group's of the first: eight side by side
                    const auto lo = __builtin_amdgcn_permlane16_swap(next[k][0].x, next[k][1].x, false, false);
                    const auto hi = __builtin_amdgcn_permlane16_swap(next[k][0].y, next[k][1].y, false, false);
                    sum[k] += __shfl_xor(sum[k], 8, WAVE);
                    sum[k] += __shfl_xor(sum[k], 16, WAVE);
                    sum[k] += __shfl_xor(sum[k], 32, WAVE);
                    const int m = row_at(i, k), n = nt * BN + wn * 64 + (lane >> 4 & 1) * 32 + side + (lane >> 5) * 8;
                    if (here && m < M) *reinterpret_cast<uint4*>(stream.next + static_cast<size_t>(m) * N + n) = make_uint4(lo[0], hi[0], lo[1], hi[1]);
                    if (here && m < M && (lane >> 3) == k) stream.ss[static_cast<size_t>(m) * (N / 64) + nt * (BN / 64) + wn] = sum[k];
                }
            }
        }
        return;
    }

    if constexpr (EPI == TG_ROPE) {
        static_assert(TN == 4, "64 columns a wavefront");
        int pos[TM], slots[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = min(m0 + (xblock + i) / 4 * 64 + (xblock + i) % 4 * 4 + row, M - 1);
            pos[i] = rope.positions[m];
            slots[i] = rope.slots ? rope.slots[m] : -1;
        }
        const int set = nt * (BN / 64) + wn, sets = rope.hd / 64;
        if (set >= N / 64) return;
        const int head = set / sets, d = set % sets * 32 + column(0, lane >> 4);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = m0 + (xblock + i) / 4 * 64 + (xblock + i) % 4 * 4 + row;
            if (m >= M) continue;
            float a[8], b[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                a[e] = acc[i][e / 4][e % 4];
                b[e] = acc[i][2 + e / 4][e % 4];
            }
            if constexpr (NORMED) {
                const float f = factor_of(i);
#pragma unroll
                for (int e = 0; e < 8; ++e) a[e] *= f, b[e] *= f;
            }
            bf16_t* to = rope.place(m, slots[i], head);
            if (!to) continue;
            if (rope.rotates(head)) rope.turned<8>(to, d, a, b, rope.angles<8>(pos[i], d));
            else rope.plain<8>(to, d, a, b);
        }
        return;
    }
    const int cols = EPI == TG_GATED ? half : N;
    constexpr int OT = EPI == TG_GATED ? TN / 2 : TN;
    constexpr int RUN = OT < 2 * GB ? 1 : 2;                   // stores that leave a row together
    const bool upper = RUN == 2 && (lane & 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + (xblock + i) / 4 * 64 + (xblock + i) % 4 * 4 + (RUN == 2 ? row & 31 : row);
        const float f = factor_of(i);
#pragma unroll
        for (int j = 0; j < OT; j += RUN * GB) {
            const int n = nt * (BN * OT / TN) + wn * OT * 16 + column(upper ? j + GB : j, lane >> 4);
            uint4 o[RUN];
#pragma unroll
            for (int k = 0; k < RUN; ++k) {
                float v[GB * 4];
#pragma unroll
                for (int e = 0; e < GB * 4; ++e) {
                    const int b = j + k * GB + e / 4;
                    if constexpr (EPI == TG_GATED && NORMED) v[e] = act.rough(acc[i][b][e % 4] * f, acc[i][b + TN - OT][e % 4] * f);
                    else v[e] = EPI == TG_GATED ? act.rough(acc[i][b][e % 4], acc[i][b + TN - OT][e % 4]) : act.plain(acc[i][b][e % 4]);
                }
                store_packed<OUT, GB * 4>(reinterpret_cast<OUT*>(&o[k]), v);
            }
            if constexpr (RUN == 2) rows_together(o[0], o[1], upper);
            if (n >= cols) continue;
#pragma unroll
            for (int k = 0; k < RUN; ++k)
                if (m + 32 * k < M) *reinterpret_cast<uint4*>(out + static_cast<size_t>(m + 32 * k) * cols + n) = o[k];
        }
    }
}

struct WideArgs {
    const bf16_t *x, *w;
    void* out;
    int M, N, K, f32;
    GatedUnit act;
    RopeStore rope;
    StreamStore stream;
    RowNorm norm;
};

template <int BM, int BN, int WM, int WN, int DX, int DW> static int launch_wide(int epi, const WideArgs& a, hipStream_t stream) {
    const int cols = epi == TG_GATED ? a.N / 2 : a.N, each = epi == TG_GATED ? BN / 2 : BN, mt = (a.M + BM - 1) / BM, nt = (cols + each - 1) / each;
#define WIDE_LAUNCH(EPI, OUT, NORMED) wide_gemm_kernel<BM, BN, WM, WN, DX, DW, EPI, OUT, NORMED><<<mt * nt, WM * WN * WAVE, 0, stream>>>(a.x, a.w, \
        static_cast<OUT*>(a.out), a.M, a.N, a.K, mt, nt, a.act, a.rope, a.stream, a.norm)
    if constexpr (BM == 64) {                                 // (few rows of plain products)
        if (epi != TG_STORE) return static_cast<int>(hipErrorInvalidValue);
        if (a.f32) WIDE_LAUNCH(TG_STORE, float, false);
        else WIDE_LAUNCH(TG_STORE, bf16_t, false);
        return NI_LAUNCH_RESULT();
    } else {
    if (epi == TG_GATED) {
        if (a.norm.ss) WIDE_LAUNCH(TG_GATED, bf16_t, true);
        else WIDE_LAUNCH(TG_GATED, bf16_t, false);
        return NI_LAUNCH_RESULT();
    }
    if constexpr (DX == 2 && BM == 128) return static_cast<int>(hipErrorInvalidValue);      // (a tile that only products with SwiGLU take)
    else if (epi == TG_ROPE && a.norm.ss) WIDE_LAUNCH(TG_ROPE, bf16_t, true);
    else if (epi == TG_ROPE) WIDE_LAUNCH(TG_ROPE, bf16_t, false);
    else if (epi == TG_STREAM) WIDE_LAUNCH(TG_STREAM, float, false);
    else if (a.f32) WIDE_LAUNCH(TG_STORE, float, false);
    else WIDE_LAUNCH(TG_STORE, bf16_t, false);
    return NI_LAUNCH_RESULT();
    }
#undef WIDE_LAUNCH
}

static int launch_wide_tile(int tile, int epi, const WideArgs& a, void* stream) {
    if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.K % 64 || static_cast<long>(a.M) * a.K >= 1l << 30 || static_cast<long>(a.N) * a.K >= 1l << 30 ||
        (reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.w) | reinterpret_cast<uintptr_t>(a.out)) % 16 ||
        (a.norm.ss && (a.norm.parts <= 0 || a.norm.parts % 4 || a.norm.parts > 64 || reinterpret_cast<uintptr_t>(a.norm.ss) % 16)))
        return static_cast<int>(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    switch (tile) {
        case 0: return launch_wide<256, 256, 2, 4, 2, 3>(epi, a, s);
        case 1: return launch_wide<128, 256, 2, 4, 3, 3>(epi, a, s);
        case 2: return launch_wide<256, 128, 4, 2, 3, 3>(epi, a, s);
        case 3: return launch_wide<128, 128, 4, 2, 5, 5>(epi, a, s);
        case 4: return launch_wide<128, 128, 2, 2, 2, 3>(epi, a, s);
        case 5: return launch_wide<64, 128, 2, 2, 3, 3>(epi, a, s);
        case 6: return launch_wide<64, 256, 2, 4, 3, 3>(epi, a, s);
        default: return static_cast<int>(hipErrorInvalidValue);
    }
}

// tile: 0 = 256 x 256, 1 = 128 x 256, 2 = 256 x 128, 3 = 128 x 128 (rows of x, rows of W), gated also 4 = 128 x 128, two a unit, plain also
// 5 = 64 x 128, two a unit, and 6 = 64 x 256.  f32: float32 results.  ss (gated; or null): the rows' sums of squares in `parts` parts, by whose root mean square with eps the rows of x are divided
NI_EXPORT int ni_wide_gemm(const void* x, const void* w, void* out, int M, int N, int K, int tile, int gated, int f32, int activation, int squared, const void* ss,
                           int parts, float eps, void* stream) {
    if (N % (gated ? 32 : 16) || (gated && (f32 || squared)) || (ss && !gated)) return static_cast<int>(hipErrorInvalidValue);
    WideArgs a{};
    a.x = static_cast<const bf16_t*>(x);
    a.w = static_cast<const bf16_t*>(w);
    a.out = out;
    a.M = M;
    a.N = N;
    a.K = K;
    a.f32 = f32;
    a.act = GatedUnit::of(activation);
    a.act.squared = squared != 0;
    a.norm = RowNorm{static_cast<const float*>(ss), parts, eps};
    return launch_wide_tile(tile, gated ? TG_GATED : TG_STORE, a, stream);
}

// h [M, N] += x . w^T; with `next` (and the weight of the norm that follows) next = h * weight and ss [M, N / 64] the sums of h^2
NI_EXPORT int ni_wide_stream(const void* x, const void* w, void* h, const void* weight, void* next, void* ss, int M, int N, int K, int tile, void* stream) {
    if (N % 64 || !h || (next && (!weight || !ss)) || (reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(next)) % 16)
        return static_cast<int>(hipErrorInvalidValue);
    WideArgs a{};
    a.x = static_cast<const bf16_t*>(x);
    a.w = static_cast<const bf16_t*>(w);
    a.out = h;
    a.M = M;
    a.N = N;
    a.K = K;
    a.stream = StreamStore{static_cast<float*>(h), static_cast<const float*>(weight), static_cast<bf16_t*>(next), static_cast<float*>(ss)};
    return launch_wide_tile(tile, TG_STREAM, a, stream);
}

// The product with the stacked matrix [q; k; v] of (H + 2 KVH) heads of hd (whole sets of 64): rotated queries to q, keys and values to the pools
NI_EXPORT int ni_wide_qkv_rope(const void* x, const void* w, void* q, const void* positions, const void* cos_t, const void* sin_t, const void* slots, void* kpool,
                               void* vpool, int M, int K, int H, int KVH, int hd, int page_size, int tile, const void* ss, int parts, float eps, void* stream) {
    if (H <= 0 || KVH <= 0 || hd <= 0 || hd % 64 || page_size <= 0 || !q || !positions || !cos_t || !sin_t || (slots && (!kpool || !vpool)) ||
        (reinterpret_cast<uintptr_t>(kpool) | reinterpret_cast<uintptr_t>(vpool) | reinterpret_cast<uintptr_t>(cos_t) | reinterpret_cast<uintptr_t>(sin_t)) % 16)
        return static_cast<int>(hipErrorInvalidValue);
    WideArgs a{};
    a.x = static_cast<const bf16_t*>(x);
    a.w = static_cast<const bf16_t*>(w);
    a.out = q;
    a.M = M;
    a.N = (H + 2 * KVH) * hd;
    a.K = K;
    a.rope = RopeStore{(const int32_t*)positions, (const float*)cos_t, (const float*)sin_t, (const int32_t*)slots, (bf16_t*)q, (bf16_t*)kpool, (bf16_t*)vpool,
                       H, KVH, hd, page_size};
    a.norm = RowNorm{static_cast<const float*>(ss), parts, eps};
    return launch_wide_tile(tile, TG_ROPE, a, stream);
}
