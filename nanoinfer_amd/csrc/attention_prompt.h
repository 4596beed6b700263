// The prompt kernel of attention_mfma.hip for head sizes 64 and 128 and pages of a power of two of tokens, sixteen or more (eight at 128): the
// same tiles, blocks, groups, rows and products as mfma_attention_kernel there, which the other head sizes and pages keep.  What is different:
//
// Keys and values go from memory straight into LDS, a page's rows by one wavefront, whose page number and addresses are scalars: no vector
// instruction works out where rows lie (sixteen a set of 32 keys there) and no row waits in registers (219 of them at most, 253 there).
// Stages go through a ring of three slots: the one whose scores are taken, the one before it, whose values are still read, and one on its way (two where
// a walk starts); the next tile's first are asked for while this one's last are multiplied.
//
// Inside the key range of all its rows a set of 32 keys is not looked at for scores that rise above the row's reference (four maxima, a
// comparison and a branch a block there): the reference is the largest score of the tile's first set (with a window: of its first sets), and
// float32 holds sums of weights up to 2^100 of it as exactly as any (an exponent of 100 is rounded by 2^-18 of the weight, which keeps eight
// bits; what such a sum is merged with and loses lies 2^-26 below it).  What leaves that range, or is not finite, is seen in the sums at the
// end of the tile, and the whole workgroup makes the tile again with a look at every set (references that move, as in the other kernel).
// That costs a second, slower walk, for scores that rise by 69 (natural units) above a first set's, or values that are no numbers.  Where it happens
// to every tile, mfma_attention_kernel : this without it : with it, us: 1,999 tokens at head size 64 39 : 37 : 77, at 128 80 : 60 : 139; 2,048 at 8,192
// 188 : 161 : 408, 420 : 335 : 892.  (A limit of 2^40 had sent scores that rise by 28 that way, which differ no more in their error against 64 bits.)
//
// The scores of a set are taken while the set before it gets its weights (at head size 128 a step of 32 keys is 25 % faster by it), so that the
// matrix cores work beside the vector unit's exponentials.  At the ends of a walk, and where scores are looked at, head size 64 takes a stage's two
// sets side by side: one at a time, short walks were slower than mfma_attention_kernel's (128 tokens at 228 keys 7.5 us there, 8.4 one at a time, 7.5
// side by side; 16 heads on 16, 256 at 256 7.4, 8.6, 7.7; 512 at 512 10.2, 10.5, 9.6).
//
// What bounds it: at long key ranges neither of the two (matrix cores busy 41 %, the vector unit 50 % of the cycles, two wavefronts a SIMD with
// a chain of instructions each); in one prompt of 2,000 tokens starts and ends: of 79,000 cycles of a workgroup's two tiles 9,000 passed before the first
// keys were there, 8,000 between the tiles, 5,000 behind the last (75,000 in all with a stage's sets side by side).
//
// Measured, mfma_attention_kernel : this, us: 32 heads of 64 on 8, 512 tokens at 512 / 1,024 keys 10.5 : 9.6, 14.9 : 13.2; 700 at 700 16.3 : 13.9; 1,024 at
// 1,024 / 4,096 18.5 : 16.6, 54.6 : 48.2; 1,999 at 1,999 38.3 : 33.8; 4,096 at 4,096 106.4 : 88.5; 2,048 at 8,192 / 32,768 170.7 : 142.8, 689.4 : 575.5;
// 24 of 128 on 8, 256 at 256 11.9 : 10.3; 512 at 512 / 2,048 17.3 : 14.9, 41.8 : 32.1; 1,999 at 1,999 75.1 : 54.5; 2,048 at 8,192 423.7 : 305.5.  Behind it
// by 2 to 4 % are few tokens of head size 64 at 1,500 to 2,000 keys in runs (100 at 2,000 15.6 : 16.0) and 256 of 16 heads on 16 (7.4 : 7.7).
//
// A single token beside the portions of a step walked its keys by one wavefront of four, as long as the portions' tiles: its four wavefronts
// now share them out as in the kernel for single tokens (attend_token), where it has a workgroup to itself.  481 tokens beside 31 with 100 to 1,100
// keys 18.6 : 14.4 us.
#pragma once
#include "lds_load.h"

#define PA_RING 3          // stages of keys and values in LDS: the current one, the one before it and one on its way

// 2 KB of K and 2 KB of V straight into LDS at k_to and v_to, sixteen bytes a lane: lane l brings the bytes at lane offset k0 (and k1, 1,024 bytes
// further on, where they also land).  Addresses in scalar registers are the same in all lanes.  (In assembly: behind the builtin every read of
// LDS waits for all such loads, whatever they write.  Whoever calls this counts them: four of vmcnt.)
__device__ __forceinline__ void load_rows_to_lds(const char* k, const char* v, uint32_t k_to, uint32_t v_to, int k0, int k1, int v0, int v1) {
    asm volatile(
        "s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %4, %0\n\tglobal_load_lds_dwordx4 %5, %0 offset:1024\n\t"
        "s_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %6, %1\n\tglobal_load_lds_dwordx4 %7, %1 offset:1024"
        ::"s"(k), "s"(v), "s"(k_to), "s"(v_to), "v"(k0), "v"(k1), "v"(v0), "v"(v1)
        : "m0");
}

// A barrier that waits for LDS only, not for loads on their way
__device__ __forceinline__ void lds_meet() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_waitcnt(0xc07f);                      // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ uint32_t lds_address(const void* p) {
    typedef __attribute__((address_space(3))) const char lds_char;
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_char*)p));
}

template <int CB, int GROUPS>
__global__ __launch_bounds__(GROUPS * MA_WAVES * WAVE) __attribute__((amdgpu_waves_per_eu(2)))
void prompt_attention_kernel(
    const bf16_t* __restrict__ q, int q_stride, const bf16_t* __restrict__ kpool, const bf16_t* __restrict__ vpool,
    const int32_t* __restrict__ block_table, int table_stride, const QTile* __restrict__ tiles,
    int n_tiles, bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml, int H, int KVH, int G,
    int chunks, int page_shift, int hpt_shift, int window, float scale, int nsplit) {
    constexpr int HD = HEAD_DIM;
    static_assert(HD == 64 || HD == 128, "whole lines a row");
    constexpr int MA_THREADS = MA_WAVES * WAVE;
    constexpr int KK = HD / 32, DT = HD / 16;
    constexpr int SUB = HD == 64 ? 2 : 1;             // sets of 32 keys a stage
    constexpr int KEYS = SUB * KSTEP;                 // keys a stage
    constexpr int ROW = HD * 2, PIECES = ROW / 16;    // bytes of a key's row, and the pieces of sixteen in it
    constexpr int CHUNK = 1024 / ROW;                 // rows that one load of a wavefront brings
    constexpr int LOADS = KEYS / CHUNK / MA_WAVES;    // of K a wavefront and stage, and as many of V
    constexpr int OWN = LOADS * CHUNK;                // rows that a wavefront brings of a stage, in one page
    static_assert(LOADS == 2, "load_rows_to_lds");
    constexpr int PAGES = GROUPS == 1 ? 3072 : 1024;  // pages of a tile whose numbers wait in LDS; those behind them are read from memory
    struct Stage { char k[KEYS * ROW], v[KEYS * ROW]; };
    __shared__ __attribute__((aligned(1024))) Stage ring[GROUPS][PA_RING];
    __shared__ __attribute__((aligned(16))) int32_t tbl[2][PAGES];
    __shared__ __attribute__((aligned(16))) floatx4_t meet_o[GROUPS][GROUPS > 1 ? MA_WAVES * CB * DT / 2 : 1][WAVE];
    __shared__ float2 meet_ml[GROUPS][GROUPS > 1 ? MA_WAVES * CB : 1][WAVE];
    __shared__ int32_t again[2][GROUPS * MA_WAVES];

    const int group = GROUPS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / MA_THREADS) : 0;
    const int tid = threadIdx.x % MA_THREADS;                 // within the group
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int r = lane % 16, kg = lane / 16;
    auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };      // (divisions go through vector registers)
    const int hpt = 1 << hpt_shift;
    const int g = chunks == 1 ? blockIdx.y : uniform(blockIdx.y / chunks), chunk = blockIdx.y - g * chunks;
    const int hh = (chunk << hpt_shift) + (r & (hpt - 1)), head = g * G + hh;
    const int tok_per_block = 16 >> hpt_shift;
    const int page_size = 1 << page_shift;
    const float scale2 = scale * LOG2E;

    // The tiles come sorted by the keys they walk, longest first; workgroup w takes tiles w, 2P-1-w, 2P+w, ... (as mfma_attention_kernel does)
    auto tile_of = [&](int round) {
        int at = (round & 1) ? (round + 1) * gridDim.x - 1 - blockIdx.x : round * gridDim.x + blockIdx.x;
        if (n_tiles <= static_cast<int>(gridDim.x) && 2 * blockIdx.y >= gridDim.y && gridDim.y > 1) at = n_tiles - 1 - at;
        return at >= n_tiles || at < 0 ? -1 : at;
    };
    // A tile as a group walks it.  All of a workgroup's groups pass the same number of stages; `own` counts the sets of 32 keys that are this
    // group's, which may be fewer or none (it then looks at the last key's row and multiplies nothing).
    struct Walk { int seq, row0, ntok, pos0, lo, last, first, stages, own, page0, pages; };
    auto walk_of = [&](const QTile& t) {
        Walk w{};
        w.seq = uniform(t.seq), w.row0 = uniform(t.row0);
        w.ntok = uniform(t.ntok), w.pos0 = uniform(t.pos0);
        const int kend = w.pos0 + w.ntok;
        w.lo = window > 0 ? max(0, w.pos0 + 1 - window) : 0;      // keys before it may lie in pages that a window has given back
        const int kbeg = w.lo / KEYS * KEYS, all = (kend - kbeg + KEYS - 1) / KEYS;
        const int per_split = nsplit == 1 ? all : uniform((all + nsplit - 1) / nsplit);
        const int run_begin = blockIdx.z * per_split, run_end = max(run_begin, min(all, run_begin + per_split));
        w.stages = (run_end - run_begin + GROUPS - 1) / GROUPS;
        const int mine = run_begin + group * w.stages;
        w.first = kbeg + mine * KEYS;
        w.own = max(0, (min(kend, kbeg + min(run_end, mine + w.stages) * KEYS) - w.first + KSTEP - 1) / KSTEP);
        w.last = min(kend, kbeg + run_end * KEYS) - 1;            // of the run
        w.page0 = (kbeg + run_begin * KEYS) >> page_shift;
        w.pages = w.stages > 0 ? min(PAGES, (w.last >> page_shift) - w.page0 + 1) : 0;
        return w;
    };
    auto load_table = [&](const Walk& w, int par) {
        const int32_t* from = block_table + static_cast<size_t>(w.seq) * table_stride + w.page0;
        for (int i = threadIdx.x; i < w.pages; i += GROUPS * MA_THREADS) tbl[par][i] = from[i];
    };
    // Q as the B operand: lane (row r, group kg) holds dims kk*32 + kg*8 .. +8; in the place of rows that are not there, some that are
    auto load_q = [&](const Walk& w, u32x4_t (&dst)[CB][KK]) {
        int head_ = head;
        asm volatile("" : "+v"(head_));                      // (addresses that are worked out here, not before the loop over tiles and kept)
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int tt = (wave * CB + c) * tok_per_block + (r >> hpt_shift);
            const bool ok = tt < w.ntok && hh < G;
            const bf16_t* from = q + static_cast<size_t>(w.row0 + (ok ? tt : 0)) * q_stride + static_cast<size_t>(ok ? head_ : 0) * HD + kg * 8;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) dst[c][kk] = *reinterpret_cast<const u32x4_t*>(from + kk * 32);
        }
    };

    // Rows lie in LDS without gaps, as a load leaves them; which piece of a row stands where is turned round by the row's number, for K so that
    // the sixteen rows of a read of sixteen bytes, and for V so that the eight rows of 32 bytes of a transposing read, meet no bank twice.
    auto turn_k = [](int row) { return HD == 64 ? (row >> 1) & 7 : row & 15; };
    auto turn_v = [](int row) { return HD == 64 ? (row >> 1 & 3) << 1 : (row & 7) << 1; };
    int piece_k[LOADS], piece_v[LOADS];
    const int line = lane / PIECES;                           // this lane's row of a load
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave * LOADS + i) * CHUNK + line;
        piece_k[i] = ((lane % PIECES) ^ turn_k(row)) * 16 + (i == 0 ? 1024 : 0);
        piece_v[i] = ((lane % PIECES) ^ turn_v(row)) * 16 + (i == 0 ? 1024 : 0);
    }
    int at_k[KK], at_v[DT];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) at_k[kk] = r * ROW + ((kk * 4 + kg) ^ turn_k(r)) * 16;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        const int row = 4 * kg + (r >> 2);
        at_v[dt] = row * ROW + ((dt * 2 + (r >> 1 & 1)) ^ turn_v(row)) * 16 + (r & 1) * 8;
    }

    int round = 0, par = 0;
    Walk cur{}, nxt{};
    bool more;                                               // nxt is a tile
    u32x4_t qf[CB][KK];
    {
        const int at = tile_of(0), at1 = tile_of(1);
        if (at < 0) return;
        more = at1 >= 0;
        const QTile t = tiles[at], t1 = tiles[more ? at1 : at];
        if constexpr (GROUPS == 1) {
            // A single token beside the portions of a step, in a workgroup of its own: its wavefronts share out its keys
            static_assert(MA_WAVES == DEC_WAVES && sizeof(ring) >= sizeof(uint16_t[DEC_WAVES][KSTEP][DEC_VROW]) + sizeof(float[DEC_WAVES][16][2]));
            if (!more && uniform(t.ntok) == 1) {
                auto vs = reinterpret_cast<uint16_t(*)[KSTEP][DEC_VROW]>(&ring[0][0]);
                attend_token<true, PAGES>(q, q_stride, kpool, vpool, block_table, table_stride, out, part_o, part_ml, H, KVH, page_size, page_shift, window, scale,
                                          nsplit, blockIdx.z, uniform(t.row0), uniform(t.seq), uniform(t.pos0), G, g, chunk, hpt, vs,
                                          reinterpret_cast<float(*)[16][2]>(vs + DEC_WAVES), tbl[0]);
                return;
            }
        }
        cur = walk_of(t);
        nxt = walk_of(t1);
        load_q(cur, qf);
        load_table(cur, 0);
        if (more) load_table(nxt, 1);
        __syncthreads();
    }
    // The stages of all tiles go through the ring one behind the other.  What is asked for is this wavefront's rows of a stage, of tile cur or
    // (in_next) nxt; where they lie outside the keys that may be read, the nearest of those instead.
    struct In { int key, left, lo, last, from_lo, from_last, page0, tbl; const int32_t* table; } in;
    bool in_next = false;
    auto enter = [&](const Walk& w, int p) {
        in = In{w.first + wave * OWN, w.stages, w.lo, w.last, w.lo & -OWN, w.last & -OWN, w.page0, p * PAGES, block_table + static_cast<size_t>(w.seq) * table_stride};
    };
    constexpr int SLOT = sizeof(Stage), LAST_SLOT = (PA_RING - 1) * SLOT;
    const uint32_t ring_at = lds_address(&ring[group][0]) + wave * LOADS * 1024;
    int slot_in = 0, slot_out = 0, ahead = 0;                // bytes into the ring; stages asked for and not taken yet
    const char *k_pool = reinterpret_cast<const char*>(kpool) - 1024, *v_pool = reinterpret_cast<const char*>(vpool) - 1024;
    int page = 0, from = 0;
    bool asks = false;                                       // there are rows to be asked for: of `page`, from key `from` on
    auto find = [&]() {
        if (in.left == 0 && !in_next && more) {
            in_next = true;
            enter(nxt, par ^ 1);
        }
        asks = in.left > 0;
        if (!asks) return;
        from = min(max(in.key, in.from_lo), in.from_last);
        const int idx = from >> page_shift;
        if (idx - in.page0 < PAGES) {
            page = tbl[0][in.tbl + idx - in.page0];
        } else {
            asm volatile("s_load_dword %0, %1, 0\n\ts_waitcnt lgkmcnt(0)" : "=s"(page) : "s"(in.table + idx));
        }
    };
    auto ask = [&]() {
        // the first row of the group's in the pool: its number fits 32 bits (the host checks the pool's size), and the lanes count from there
        const uint32_t row = ((static_cast<uint32_t>(max(uniform(page), 0)) * KVH + g) << page_shift) + (from & (page_size - 1));
        const size_t at = static_cast<size_t>(row) * ROW;
        const uint32_t to = ring_at + slot_in;
        const int key = in.key - from, lo = in.lo - from, last = in.last - from;
        const int key0 = min(max(key + line, lo), last), key1 = min(max(key + line + CHUNK, lo), last);
        // (the pools' addresses are 1,024 bytes before them, and so much is in the lanes' places: a load that lands so much further on reads there)
        load_rows_to_lds(k_pool + at, v_pool + at, to, to + KEYS * ROW, key0 * ROW + piece_k[0], key1 * ROW + piece_k[1], key0 * ROW + piece_v[0],
                         key1 * ROW + piece_v[1]);
        in.key += KEYS;
        --in.left;
        ++ahead;
        slot_in = slot_in == LAST_SLOT ? 0 : slot_in + SLOT;
    };
    auto fill = [&]() {                                      // where nobody reads the ring: two stages on their way, if there are any, and the next to ask for
        find();
        while (ahead < 2 && asks) {
            ask();
            find();
        }
    };
    // this wavefront's loads of the next stage to take have landed (a stage behind it is on its way only where a walk starts)
    auto landed = [&]() {
        if (ahead > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };
    enter(cur, 0);
    fill();

    bool safe = false;                                       // the tile is made again, every step with a look at its largest scores
    for (;;) {
        int hi[CB], lo_max = 0, p_min = 1 << 30;       // of all blocks: the latest first key and the earliest position
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int tb0 = (wave * CB + c) * tok_per_block, tt = tb0 + (r >> hpt_shift);
            hi[c] = tt < cur.ntok && hh < G ? cur.pos0 + tt : -1;        // the row's position; -1 where there is none
            if (tb0 < cur.ntok) p_min = min(p_min, cur.pos0 + tb0);
            if (window > 0 && tb0 < cur.ntok) lo_max = max(lo_max, cur.pos0 + min(cur.ntok, tb0 + tok_per_block) - window);
        }
        const int own = wave * CB * tok_per_block < cur.ntok ? cur.own : 0;      // a wavefront without rows multiplies nothing
        // the sets [in_lo, in_hi) lie inside the key range of every row of this wavefront
        const int in_lo = lo_max > cur.first ? (lo_max - cur.first + KSTEP - 1) / KSTEP : 0;
        const int in_hi = p_min - (KSTEP - 1) >= cur.first ? min(own, (p_min - (KSTEP - 1) - cur.first) / KSTEP + 1) : 0;
        bool primed = false;                                 // every row has a reference

        float m_run[CB];
        floatx4_t o[CB][DT], l_run[CB];
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            m_run[c] = NEG_BIG;
            l_run[c] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[c][dt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
        }
        // S^T of the 32 keys whose rows start at k: this lane's row of every block, keys t*16 + kg*4 + i
        auto scores = [&](const char* k, floatx4_t (&sc)[CB][2]) {
            u32x4_t ka[2][KK];
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) ka[t][kk] = *reinterpret_cast<const u32x4_t*>(k + at_k[kk] + t * 16 * ROW);
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    sc[c][t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int kk = 0; kk < KK; ++kk)
                        sc[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ka[t][kk]), __builtin_bit_cast(bf16x8_t, qf[c][kk]), sc[c][t], 0, 0, 0);
                }
        };
        // O^T += V^T . P^T; V^T as the A operand (read_v_operand)
        auto add_values = [&](const char* v, const uint4 (&pf)[CB]) {
            typedef __attribute__((address_space(3))) shortx4_t* lds_ptr;
            u32x4_t vf[DT];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const uint2 a = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(v + at_v[dt])));
                const uint2 b = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(v + at_v[dt] + 16 * ROW)));
                vf[dt] = u32x4_t{a.x, a.y, b.x, b.y};
            }
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                l_run[c] = row_sum_step(pf[c], l_run[c]);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
                    o[c][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, vf[dt]), __builtin_bit_cast(bf16x8_t, pf[c]), o[c][dt], 0, 0, 0);
            }
        };
        // n neighbouring sets of a stage, with a look at how far their scores rise (key0: this lane's first key of them):
        auto any_sets = [&](auto N, const char* k, const char* v, int key0) {
            constexpr int n = decltype(N)::value;
            floatx4_t sc[n][CB][2];
#pragma unroll
            for (int s = 0; s < n; ++s) scores(k + s * KSTEP * ROW, sc[s]);
            float raw[n][CB][8], lane_max[CB];
            bool risen = false;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                const int lo = window > 0 ? hi[c] + 1 - window : 0;
                lane_max[c] = NEG_BIG;
#pragma unroll
                for (int s = 0; s < n; ++s) lane_max[c] = fmaxf(lane_max[c], mask_scores<true>(sc[s][c], key0 + s * KSTEP, lo, hi[c], true, raw[s][c]));
                risen = risen || above_reference(lane_max[c], scale2, m_run[c]);
            }
            if (__any(risen)) {
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    const float corr = move_reference(lane_max[c], scale2, m_run[c]);
                    l_run[c] *= corr;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) o[c][dt] *= corr;
                }
            }
            uint4 pf[n][CB];
#pragma unroll
            for (int s = 0; s < n; ++s)
#pragma unroll
                for (int c = 0; c < CB; ++c) pf[s][c] = weights<true>(raw[s][c], scale2, m_run[c]);
#pragma unroll
            for (int s = 0; s < n; ++s) add_values(v + s * KSTEP * ROW, pf[s]);
            if (!primed) {
                bool cold = safe;
#pragma unroll
                for (int c = 0; c < CB; ++c) cold = cold || (hi[c] >= 0 && m_run[c] <= 0.5f * NEG_BIG);
                primed = !__any(cold);
            }
        };
        // Without a window: a tile's first sets, from the largest scores of the first of which the rows take their references, and those with keys
        // behind some rows' positions.
        auto edge_sets = [&](auto N, const char* k, const char* v, int key0) {
            constexpr int n = decltype(N)::value;
            floatx4_t sc[n][CB][2];
#pragma unroll
            for (int s = 0; s < n; ++s) scores(k + s * KSTEP * ROW, sc[s]);
            if (!primed) {
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    float mx = fmaxf(sc[0][c][0][0], sc[0][c][1][0]);
#pragma unroll
                    for (int i = 1; i < 4; ++i) mx = fmaxf(mx, fmaxf(sc[0][c][0][i], sc[0][c][1][i]));
                    m_run[c] = row_max4(mx) * scale2;
                }
                primed = true;
            }
            uint4 pf[n][CB];
#pragma unroll
            for (int s = 0; s < n; ++s)
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    float w[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        w[i] = __builtin_amdgcn_exp2f(fmaf(sc[s][c][i / 4][i % 4], scale2, -m_run[c]));
                        w[i] = key0 + s * KSTEP + i / 4 * 16 + i % 4 <= hi[c] ? w[i] : 0.f;
                    }
                    pf[s][c] = make_uint4(pack_bf16x2(w[0], w[1]), pack_bf16x2(w[2], w[3]), pack_bf16x2(w[4], w[5]), pack_bf16x2(w[6], w[7]));
                }
#pragma unroll
            for (int s = 0; s < n; ++s) add_values(v + s * KSTEP * ROW, pf[s]);
        };
        // A set whose keys lie inside the range of every row, once every row has a reference: its scores have been taken, and those of the set
        // behind it (whose rows start at k) are, while it gets its weights and its values.
        floatx4_t sc[2][CB][2];
        auto inner_set = [&](auto P, const char* k, const char* v) {
            constexpr int p = decltype(P)::value;
            scores(k, sc[p ^ 1]);
            uint4 pf[CB];
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                float raw[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) raw[i] = sc[p][c][i / 4][i % 4];
                pf[c] = weights<false>(raw, scale2, m_run[c]);
            }
            add_values(v, pf);
        };
        if (ahead == 0) fill();                              // (behind a tile without stages)
        int met = 0;
        const char *here = nullptr, *before = nullptr;       // the rows of the stage met last, and of the one before it
        auto meet = [&]() {                                  // the next stage: it has landed for everybody, and everybody is done with the last but one
            landed();
            lds_meet();
            --ahead;
            ++met;
            before = here;
            here = reinterpret_cast<const char*>(&ring[group][0]) + slot_out;
            slot_out = slot_out == LAST_SLOT ? 0 : slot_out + SLOT;
            if (ahead == 0) {
                if (asks) ask();
                find();
            }
        };
        constexpr int VALUES = KEYS * ROW, SET = KSTEP * ROW;
        for (int j = 0; j < own;) {
            if (met <= j / SUB) meet();
            if (primed && j % SUB == 0 && j >= in_lo && j + 2 < in_hi) {
                scores(here, sc[0]);
                do {                                         // two sets a turn, as their registers change places
                    if constexpr (SUB == 2) {
                        inner_set(Index<0>{}, here + SET, here + VALUES);
                        meet();
                        inner_set(Index<1>{}, here, before + VALUES + SET);
                    } else {
                        meet();
                        inner_set(Index<0>{}, here, before + VALUES);
                        meet();
                        inner_set(Index<1>{}, here, before + VALUES);
                    }
                    j += 2;
                } while (j + 2 < in_hi);                     // (the last scores are taken again)
            } else {
                const char* k = here + j % SUB * SET;
                const int key0 = cur.first + j * KSTEP + kg * 4;
                // (both sets of a stage side by side: one alone is a chain of instructions that nothing covers)
                const bool look = safe || window > 0 || !(primed || (j == 0 && in_hi > 0));
                if (SUB == 2 && j % SUB == 0 && j + 1 < own) {
                    if (look) any_sets(Index<SUB>{}, k, k + VALUES, key0);
                    else edge_sets(Index<SUB>{}, k, k + VALUES, key0);
                    j += 2;
                } else {
                    if (look) any_sets(Index<1>{}, k, k + VALUES, key0);
                    else edge_sets(Index<1>{}, k, k + VALUES, key0);
                    ++j;
                }
            }
        }
        while (met < cur.stages) meet();

        // Sets without a look at their scores: where one has risen so far that weights or sums are no longer numbers in range (or never
        // were), everybody makes the tile again with one.
        {
            bool bad = false;
            if (!safe) {
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    float zero = 0.f;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) zero = fmaf(o[c][dt][i], 0.f, zero);
                    bad = bad || (hi[c] >= 0 && !(l_run[c][0] < 0x1p100f && zero == 0.f));
                }
            }
            again[round & 1][group * MA_WAVES + wave] = __any(bad);
        }
        if constexpr (GROUPS > 1) {
            // Each group finishes one half of the dims and hands over the other.  (Where a tile has no stages, no barrier stands between the
            // reads of the tile before and these writes.)
            if (cur.stages == 0) __syncthreads();
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                meet_ml[group][wave * CB + c][lane] = make_float2(m_run[c], l_run[c][0]);
#pragma unroll
                for (int dt = 0; dt < DT / 2; ++dt) meet_o[group][(wave * CB + c) * (DT / 2) + dt][lane] = group == 0 ? o[c][DT / 2 + dt] : o[c][dt];
            }
        }
        lds_meet();
        if (__any(lane < GROUPS * MA_WAVES && again[round & 1][lane % (GROUPS * MA_WAVES)])) {
            safe = true;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();                                 // nobody's load is on its way, nobody reads a flag any more
            ahead = 0;
            slot_in = slot_out;
            in_next = false;
            enter(cur, par);
            fill();
            continue;
        }
        if (more) load_q(nxt, qf);                           // (asked for before the stores below)
        {
            int kg_ = kg, head_ = head;                      // (addresses that are worked out here, not before the loop over tiles and kept)
            asm volatile("" : "+v"(kg_), "+v"(head_));
            constexpr int MINE = GROUPS > 1 ? DT / 2 : DT;
            const int dim0 = group * MINE * 16 + kg_ * 4;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                float l = l_run[c][0], m = m_run[c];
                floatx4_t done[MINE];
#pragma unroll
                for (int dt = 0; dt < MINE; ++dt) done[dt] = GROUPS > 1 && group == 1 ? o[c][DT - MINE + dt] : o[c][dt];
                if constexpr (GROUPS > 1) {
                    const float2 other = meet_ml[group ^ 1][wave * CB + c][lane];
                    m = fmaxf(m, other.x);
                    const float mine = __builtin_amdgcn_exp2f(m_run[c] - m), theirs = __builtin_amdgcn_exp2f(other.x - m);
                    l = l * mine + other.y * theirs;
#pragma unroll
                    for (int dt = 0; dt < MINE; ++dt) done[dt] = done[dt] * mine + meet_o[group ^ 1][(wave * CB + c) * MINE + dt][lane] * theirs;
                }
                if (hi[c] < 0) continue;
                const int row = cur.row0 + hi[c] - cur.pos0;
                if (nsplit > 1) {
                    // partial (maximum, sum, unnormalised output) of this split, merged by a second kernel
                    const size_t p = (static_cast<size_t>(row) * H + head_) * nsplit + blockIdx.z;
                    if (kg_ == 0 && group == 0) { part_ml[p * 2] = m * LN2; part_ml[p * 2 + 1] = l; }     // the merge kernel works in base e
#pragma unroll
                    for (int dt = 0; dt < MINE; ++dt)
                        *reinterpret_cast<float4*>(part_o + p * HD + dim0 + dt * 16) = make_float4(done[dt][0], done[dt][1], done[dt][2], done[dt][3]);
                } else if (l != 0.f) {                           // (no number too, so that the row is none and not what the memory held)
                    const float inv = 1.0f / l;
                    bf16_t* dst = out + static_cast<size_t>(row) * H * HD + static_cast<size_t>(head_) * HD + dim0;
#pragma unroll
                    for (int dt = 0; dt < MINE; ++dt)
                        *reinterpret_cast<uint2*>(dst + dt * 16) =
                            make_uint2(pack_bf16x2(done[dt][0] * inv, done[dt][1] * inv), pack_bf16x2(done[dt][2] * inv, done[dt][3] * inv));
                }
            }
        }
        if (!more) return;
        // the next tile, whose first stages have been asked for, and the one behind it
        ++round;
        par ^= 1;
        safe = false;
        cur = nxt;
        if (!in_next) enter(cur, par);
        in_next = false;
        const int at = tile_of(round + 1);
        more = at >= 0;
        if (more) {
            nxt = walk_of(tiles[at]);
            load_table(nxt, par ^ 1);
            __syncthreads();
        }
    }
}
