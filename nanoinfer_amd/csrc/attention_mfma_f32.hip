// Attention over the paged key/value cache on the matrix cores of gfx950, in true float32.  Compiled once per
// head size (-DHEAD_DIM=n, a multiple of 16 up to 256).  The float32 twins of the bfloat16 kernels
// of attention_mfma.hip, with the same interfaces: first the kernel for prompt portions, described here; at the end of the
// file the one for single tokens.
//
// A workgroup of four wavefronts owns one tile of consecutive tokens of one sequence (or half of one) and the query
// heads of one kv head (up to 16 at a time).  A "row" is one (token, head) pair; a wavefront owns one block of 16 rows, or
// two.  All rows of a workgroup read the same keys and values, 32 at a time.
//
// The vector unit works at the rate of the float32 matrix instructions (v_mfma_f32_16x16x4_f32, 32 cycles for four of K),
// and bfloat16 ones are sixteen times faster: every number is taken apart into three bfloat16 parts that add up to it (exactly, of 2^-110 and
// more), and six of the nine products of two such sums are made, what is left out being at most 2^-24 of a product and 2^-27 on average:
//
//   S^T[key, row]   = K[key, :] . Q[row, :]      parts of K from LDS as the A operand, of Q (scaled, split once) as B
//   softmax           float32, online; a lane holds 8 scores (keys 4*kg + i of both 16-key halves) of ONE row, so a row's
//                     maximum crosses lanes only when it has to move
//   O^T[dim, row]  += V^T[dim, key] . P^T[key, row]   a lane's eight weights, split in its registers, are the B operand;
//                     V^T comes from V's parts in LDS, which lie as in the cache, by transposing reads
//
// K and V are split once a workgroup, on their way into LDS.  The matrix instructions of 32 keys by 16 rows then take 768 cycles of a
// wavefront at head size 64 where the float32 ones took 2,048, and what bounds the kernel is the vector unit (350
// instructions a step: exponentials, the splits, addresses): two blocks a wavefront share the splits of K and V and the reads
// of LDS.  Measured, on the float32 instructions : in parts, with the merge of the runs (us): head size 64, 32 heads on 8, 512 tokens at
// 512 / 1,536 / 4,096 keys 46.5 : 26.5, 101 : 53.7, 233 : 109, 2,048 at 2,048 253 : 132; head size 128, 24 on 8, 512 at 1,536 202 : 95; head
// size 256, 8 on 2, 1,024 at 1,024 132 : 71.  Against 64 bits the results are off by 0.65 to 0.8 of what they were (1.7e-7 : 2.5e-7
// for 512 tokens at 512 keys).
//
// An infinity less itself has no rest (nor has a number so large that it rounds to one): a tile with a result that is not finite is
// made again on the float32 instructions (exact_tile), which give what a float32 product makes of such numbers.
//
// Formula (reference: src/op/kernels/cuda/prefill_attention_kernel.cu:66-141, 422-455, which
// forms the whole score matrix with two library products per chunk): the query at position P
// reads keys max(0, P+1-window)..P, scores are scaled by `scale`, softmax subtracts a reference
// and divides by the plain sum.
#include "common.h"

#ifndef HEAD_DIM
#error "HEAD_DIM must be defined"
#endif
static_assert(HEAD_DIM % 16 == 0 && HEAD_DIM >= 16 && HEAD_DIM <= 256, "head size: multiple of 16, at most 256");

typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

#define MA_WAVES 4
#define NEG_BIG (-1.0e30f)
#define ROW_PAD 4      // floats of padding per staged row: the sixteen rows of a 16-byte read fall on different banks
// How far a row's scores may rise above the reference its weights are taken against before the
// reference is moved and the output rescaled (e^5.545 = 2^8).  Softmax is the same whatever the
// reference, as long as numerator and denominator share it.
#define REF_SLACK 5.545177444479562f
// A row's reference before its first score.  A key that a row does not see scores minus infinity, and its weight against this or any
// later reference is zero by itself: keys are told apart by their places, never by their scores, so that NaN and infinities
// reach the sums whichever step they lie in.
#define LOWEST (-3.4028234663852886e38f)

struct QTile { int32_t seq, row0, ntok, pos0; };   // tokens row0..row0+ntok-1 of the batch, positions pos0..

__device__ __forceinline__ float lanes4(float x, bool take_max) {
    // over the four lanes that hold one row (lanes r, r+16, r+32, r+48): maximum or sum
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float u = __uint_as_float(a[0]), v = __uint_as_float(a[1]);
    x = take_max ? fmaxf(u, v) : u + v;
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float s = __uint_as_float(b[0]), t = __uint_as_float(b[1]);
    return take_max ? fmaxf(s, t) : s + t;
}

__device__ __forceinline__ float quads4(float x, bool take_max) {
    // over the four lanes r, r + 4, r + 8, r + 12 of sixteen (row_ror:4, then row_ror:8): maximum or sum
    float y = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, false));
    x = take_max ? fmaxf(x, y) : x + y;
    y = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false));
    return take_max ? fmaxf(x, y) : x + y;
}

struct TileArgs {
    const float *q, *kpool, *vpool;
    const int32_t* block_table;
    float *out, *part_o, *part_ml;
    int q_stride, table_stride, H, KVH, page_size, page_shift, hpt_shift, window, nsplit;
    float scale;
};

constexpr int TBL_MAX = 1024;                       // pages of a sequence that a workgroup looks up at a time
constexpr int PKEYS = 32;                           // keys of a step in three parts; a run of keys is whole steps

// One block of 16 rows a wavefront (of the `blocks` it owns) on the float32 instructions.  The k index of an MFMA is only a
// label: lane group kg of MFMA j takes dim kg*HD/4 + j of K and Q; of the second product the weight of key 4*kg + i is register i
// of the lane, and the A operand's row m stands for dim m*HD/16 + db (MFMA db), so that a lane ends up with HD/4
// consecutive dims of its row's output.
struct ExactLds {
    static constexpr int KSTEP = HEAD_DIM <= 128 ? 32 : 16;
    float k[KSTEP][HEAD_DIM + ROW_PAD], v[KSTEP][HEAD_DIM + ROW_PAD];
};

template <bool POW2>
__device__ __forceinline__ void exact_tile(const TileArgs& a, const QTile& tile, int blocks, int block, ExactLds& lds, int32_t* tbl) {
    constexpr int HD = HEAD_DIM;
    constexpr int THREADS = MA_WAVES * WAVE;
    constexpr int KSTEP = ExactLds::KSTEP;   // keys of a step
    constexpr int HALVES = KSTEP / 16;
    constexpr int QK = HD / 4;                     // MFMAs of the first product per 16 keys; floats of Q a lane holds
    constexpr int DB = HD / 16;                    // MFMAs of the second product per 4 keys
    constexpr int ROW = HD + ROW_PAD;
    auto& ksm = lds.k;
    auto& vsm = lds.v;
    const float *q = a.q, *kpool = a.kpool, *vpool = a.vpool;
    const int H = a.H, KVH = a.KVH, page_size = a.page_size, page_shift = a.page_shift, hpt_shift = a.hpt_shift, window = a.window;
    const int nsplit = a.nsplit, q_stride = a.q_stride, table_stride = a.table_stride;
    const float scale = a.scale;
    const int32_t* block_table = a.block_table;
    float *out = a.out, *part_o = a.part_o, *part_ml = a.part_ml;
    const int G = H / KVH;
    const int hpt = 1 << hpt_shift;
    const int chunks = (G + hpt - 1) >> hpt_shift;
    const int g = blockIdx.y / chunks;
    const int chunk = blockIdx.y % chunks;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int r = lane % 16, kg = lane / 16;

    // the wavefront's block of 16 rows: tokens wave*16/hpt .. of the tile, heads fastest
    const int tok_per_block = 16 >> hpt_shift;
    const int tb0 = (wave * blocks + block) * tok_per_block;
    const int tt = tb0 + (r >> hpt_shift);
    const int hh = (chunk << hpt_shift) + (r & (hpt - 1));
    const int head = g * G + hh;
    const bool row_ok = tt < tile.ntok && hh < G;
    const int pos = tile.pos0 + tt;
    const int row_lo = (row_ok && window > 0) ? max(0, pos + 1 - window) : 0;
    const bool blk_ok = tb0 < tile.ntok;                                     // uniform in the wavefront
    const int blk_pmin = tile.pos0 + tb0;
    const int blk_pmax = tile.pos0 + min(tile.ntok, tb0 + tok_per_block) - 1;
    const int blk_lo_max = window > 0 ? max(0, blk_pmax + 1 - window) : 0;

    // key range of the workgroup, walked in steps of KSTEP: the same run of PKEYS at a time as in parts_tile, since the other runs
    // of these rows may have been made there; only keys tile_lo..kend-1 are read from the cache (all of them the
    // sequence's own, none given back)
    const int kend = tile.pos0 + tile.ntok;
    const int tile_lo = window > 0 ? max(0, tile.pos0 + 1 - window) : 0;
    const int kbeg = tile_lo / PKEYS * PKEYS;
    const int per_split = ((kend - kbeg + PKEYS - 1) / PKEYS + nsplit - 1) / nsplit;
    const int kfirst = kbeg + blockIdx.z * per_split * PKEYS;
    const int nsteps = (max(0, min(kend - kfirst, per_split * PKEYS)) + KSTEP - 1) / KSTEP;

    const int32_t* table = block_table + static_cast<size_t>(tile.seq) * table_stride;
    auto page_of = [&](int key) { return POW2 ? (key >> page_shift) : key / page_size; };
    auto slot_of = [&](int key) { return POW2 ? (key & (page_size - 1)) : key % page_size; };
    int key_lo = 0, key_hi = 0, lp0 = 0;              // keys of the current table segment, and its first page
    auto row_address = [&](int key) -> size_t {       // offset of key's row for kv head g; key clamped to keys that may be read
        const int kc = min(max(key, key_lo), key_hi);
        const int page = tbl[page_of(kc) - lp0];
        return ((static_cast<size_t>(max(page, 0)) * KVH + g) * page_size + slot_of(kc)) * HD;
    };

    // Q, scaled, as the B operand: lane (row r, group kg) holds dims kg*HD/4 .. +HD/4
    float qf[QK];
    if (row_ok) {
        VecIO<float, QK>::load(q + static_cast<size_t>(tile.row0 + tt) * q_stride + static_cast<size_t>(head) * HD + kg * QK, qf);
#pragma unroll
        for (int j = 0; j < QK; ++j) qf[j] *= scale;
    } else {
#pragma unroll
        for (int j = 0; j < QK; ++j) qf[j] = 0.f;
    }

    float m_ref = LOWEST, l_lane = 0.f;       // the row's reference; the sum of this lane's own weights
    floatx4_t o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    // a step's keys are staged when its turn comes: this way is for the rare tile, and kept short
    for (int seg0 = 0; seg0 < nsteps;) {
        const int seg_first = kfirst + seg0 * KSTEP;
        lp0 = page_of(max(seg_first, tile_lo));
        const int seg_steps = min(nsteps - seg0, ((lp0 + TBL_MAX) * page_size - seg_first) / KSTEP);
        key_lo = max(seg_first, tile_lo);
        key_hi = min(seg_first + seg_steps * KSTEP, kend) - 1;
        __syncthreads();                   // nobody still reads the previous segment's table
        for (int i = tid; i <= page_of(key_hi) - lp0; i += THREADS) tbl[i] = table[lp0 + i];
#pragma nounroll
        for (int s = 0; s < seg_steps; ++s) {
            const int ks = seg_first + s * KSTEP;
            __syncthreads();               // nobody still reads the last step's keys
            for (int item = tid; item < KSTEP * HD / 4; item += THREADS) {
                const int key = item / (HD / 4), dim0 = item % (HD / 4) * 4;
                const size_t at = row_address(ks + key) + dim0;
                *reinterpret_cast<float4*>(&ksm[key][dim0]) = *reinterpret_cast<const float4*>(kpool + at);
                *reinterpret_cast<float4*>(&vsm[key][dim0]) = *reinterpret_cast<const float4*>(vpool + at);
            }
            __syncthreads();
            const bool act = blk_ok && ks <= blk_pmax;                           // else all rows lie before these keys
            const bool inner = act && ks >= blk_lo_max && ks + KSTEP - 1 <= blk_pmin;   // every key counts for every row
            if (act) {
                const float (*kb)[ROW] = ksm;
                const float (*vb)[ROW] = vsm;
                // 1. scores: this lane gets row r, keys ks + 16*t + 4*kg + i
                floatx4_t st[HALVES];
#pragma unroll
                for (int t = 0; t < HALVES; ++t) {
                    st[t] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j4 = 0; j4 < QK / 4; ++j4) {
                        const float4 ka = *reinterpret_cast<const float4*>(&kb[t * 16 + r][kg * QK + j4 * 4]);
                        st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.x, qf[j4 * 4 + 0], st[t], 0, 0, 0);
                        st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.y, qf[j4 * 4 + 1], st[t], 0, 0, 0);
                        st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.z, qf[j4 * 4 + 2], st[t], 0, 0, 0);
                        st[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.w, qf[j4 * 4 + 3], st[t], 0, 0, 0);
                    }
                }
                float sc[HALVES][4];
                float lane_max = -INFINITY;
#pragma unroll
                for (int t = 0; t < HALVES; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        float v = st[t][i];
                        if (!inner) {
                            const int key = ks + t * 16 + kg * 4 + i;
                            v = (row_ok && key <= pos && key >= row_lo) ? v : -INFINITY;
                        }
                        sc[t][i] = v;
                        lane_max = fmaxf(lane_max, v);
                    }
                // 2. a row whose scores have risen far above its reference: move it, rescale what was summed
                if (__any(lane_max - REF_SLACK > m_ref)) {
                    const float mx = lanes4(lane_max, true);
                    const bool move = mx > m_ref + REF_SLACK;
                    const float m_new = move ? mx : m_ref;
                    const float corr = move ? expf(m_ref - m_new) : 1.0f;
                    m_ref = m_new;
                    l_lane *= corr;
#pragma unroll
                    for (int db = 0; db < DB; ++db) o[db] *= corr;
                }
                // 3. weights, and O^T += V^T . P^T for the keys {16*t + 4*kg + i} of MFMA (t, i)
#pragma unroll
                for (int t = 0; t < HALVES; ++t)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float p = expf(sc[t][i] - m_ref);
                        l_lane += p;
                        float va[DB];
                        VecIO<float, DB>::load(&vb[t * 16 + kg * 4 + i][r * DB], va);
#pragma unroll
                        for (int db = 0; db < DB; ++db)
                            o[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[db], p, o[db], 0, 0, 0);
                    }
            }
        }
        seg0 += seg_steps;
    }

    const float l = lanes4(l_lane, false);
    if (row_ok) {
        // this lane holds dims kg*HD/4 + i*DB + db of its row in o[db][i]
        float vals[QK];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int db = 0; db < DB; ++db) vals[i * DB + db] = o[db][i];
        if (nsplit > 1) {
            const size_t p = (static_cast<size_t>(tile.row0 + tt) * H + head) * nsplit + blockIdx.z;
            if (kg == 0) { part_ml[p * 2] = m_ref; part_ml[p * 2 + 1] = l; }
            VecIO<float, QK>::store(part_o + p * HD + kg * QK, vals);
        } else {
            const float inv = 1.0f / l;
#pragma unroll
            for (int j = 0; j < QK; ++j) vals[j] *= inv;
            VecIO<float, QK>::store(out + static_cast<size_t>(tile.row0 + tt) * H * HD + static_cast<size_t>(head) * HD + kg * QK, vals);
        }
    }
}

// Eight float32 numbers as three times eight bfloat16 numbers that add up to them.
struct Parts { uint4 p[3]; };
__device__ __forceinline__ Parts parts8(const float* v) {
    uint32_t h[4], m[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
        const float r0 = v[2 * i] - __uint_as_float(h[i] << 16), r1 = v[2 * i + 1] - __uint_as_float(h[i] & 0xffff0000u);
        m[i] = pack_bf16x2(r0, r1);
        l[i] = pack_bf16x2(r0 - __uint_as_float(m[i] << 16), r1 - __uint_as_float(m[i] & 0xffff0000u));
    }
    return Parts{{make_uint4(h[0], h[1], h[2], h[3]), make_uint4(m[0], m[1], m[2], m[3]), make_uint4(l[0], l[1], l[2], l[3])}};
}

// of six products of parts, the small ones first
constexpr int PART_A[6] = {2, 0, 1, 1, 0, 0}, PART_B[6] = {0, 2, 1, 0, 1, 0};
__device__ __forceinline__ floatx4_t times(const uint4& a, const uint4& b, floatx4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

constexpr int PSLOTS = HEAD_DIM <= 64 ? 2 : 1;              // steps that LDS holds
struct PartLds {
    uint16_t k[PSLOTS][3][PKEYS][HEAD_DIM + 8], v[PSLOTS][3][PKEYS][HEAD_DIM + 8];
};

// V^T as the A operand of the second product, from a part of V as it lies in the cache: gfx950's transposing read hands lane
// (r, kg) the elements V[4 * kg + i][dim0 + r] when it gives the address of V[4 * kg + r / 4][dim0 + 4 * (r % 4)].
typedef short shortx4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 read_v_part(const uint16_t* part, int dim0, int r, int kg) {
    typedef __attribute__((address_space(3))) shortx4_t* lds_ptr;
    const uint16_t* at = part + (4 * kg + (r >> 2)) * (HEAD_DIM + 8) + dim0 + 4 * (r & 3);
    const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at)));
    const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at + 16 * (HEAD_DIM + 8))));
    return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// CB blocks of 16 rows a wavefront in three parts.  False, and nothing stored, where a result is not finite.
template <int CB, bool POW2>
__device__ __forceinline__ bool parts_tile(const TileArgs& a, const QTile& tile, PartLds& lds, int32_t* tbl) {
    constexpr int HD = HEAD_DIM, THREADS = MA_WAVES * WAVE;
    constexpr int KK = HD / 32, KC = (HD + 31) / 32;        // whole steps of 32 dims of the first product, and all (the last may be half)
    constexpr int DT = HD / 16;
    const int G = a.H / a.KVH, hpt = 1 << a.hpt_shift, chunks = (G + hpt - 1) >> a.hpt_shift;
    const int g = blockIdx.y / chunks, chunk = blockIdx.y % chunks;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int r = lane % 16, kg = lane / 16;
    const int window = a.window, page_size = a.page_size;

    const int tok_per_block = 16 >> a.hpt_shift;
    const int hh = (chunk << a.hpt_shift) + (r & (hpt - 1)), head = g * G + hh;
    int pos[CB], row_lo[CB], tt[CB], blk_pmin[CB], blk_pmax[CB], blk_lo_max[CB];
    bool row_ok[CB], blk_ok[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        const int tb0 = (wave * CB + c) * tok_per_block;
        tt[c] = tb0 + (r >> a.hpt_shift);
        row_ok[c] = tt[c] < tile.ntok && hh < G;
        pos[c] = tile.pos0 + tt[c];
        row_lo[c] = (row_ok[c] && window > 0) ? max(0, pos[c] + 1 - window) : 0;
        blk_ok[c] = tb0 < tile.ntok;
        blk_pmin[c] = tile.pos0 + tb0;
        blk_pmax[c] = tile.pos0 + min(tile.ntok, tb0 + tok_per_block) - 1;
        blk_lo_max[c] = window > 0 ? max(0, blk_pmax[c] + 1 - window) : 0;
    }
    const int kend = tile.pos0 + tile.ntok;
    const int tile_lo = window > 0 ? max(0, tile.pos0 + 1 - window) : 0;
    const int kbeg = tile_lo / PKEYS * PKEYS;
    const int nsteps_all = (kend - kbeg + PKEYS - 1) / PKEYS;
    const int per_split = (nsteps_all + a.nsplit - 1) / a.nsplit;
    const int s_begin = blockIdx.z * per_split;
    const int nsteps = max(0, min(nsteps_all, s_begin + per_split) - s_begin);
    const int kfirst = kbeg + s_begin * PKEYS;

    const int32_t* table = a.block_table + static_cast<size_t>(tile.seq) * a.table_stride;
    auto page_of = [&](int key) { return POW2 ? (key >> a.page_shift) : key / page_size; };
    auto slot_of = [&](int key) { return POW2 ? (key & (page_size - 1)) : key % page_size; };
    int key_lo = 0, key_hi = 0, lp0 = 0;              // keys of the current table segment, and its first page
    auto row_address = [&](int key) -> size_t {       // offset of key's row for kv head g; key clamped to keys that may be read
        const int kc = min(max(key, key_lo), key_hi);
        const int page = tbl[page_of(kc) - lp0];
        return static_cast<size_t>((static_cast<uint32_t>(max(page, 0)) * a.KVH + g) * page_size + slot_of(kc)) * HD;
    };

    // Q, scaled, as the B operand: lane (row r, group kg) holds dims kk * 32 + kg * 8 .. +8; of a last half step dims
    // KK * 32 + kg * 4 .. +4 in the first half of its operand, zeros in the second (of both operands)
    Parts qf[CB][KC];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        const float* qrow = a.q + static_cast<size_t>(tile.row0 + (row_ok[c] ? tt[c] : 0)) * a.q_stride + static_cast<size_t>(row_ok[c] ? head : 0) * HD;
#pragma unroll
        for (int kk = 0; kk < KC; ++kk) {
            float v[8];
            if (kk < KK) {
                VecIO<float, 8>::load(qrow + kk * 32 + kg * 8, v);
            } else {
                VecIO<float, 4>::load(qrow + KK * 32 + kg * 4, v);
#pragma unroll
                for (int j = 4; j < 8; ++j) v[j] = 0.f;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = row_ok[c] ? v[j] * a.scale : 0.f;
            qf[c][kk] = parts8(v);
        }
    }
    float m_ref[CB], l_lane[CB];
    floatx4_t o[CB][DT];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        m_ref[c] = LOWEST;
        l_lane[c] = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) o[c][dt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    }

    // Staging: a thread loads eight numbers of one key's K row and of its V row and leaves them in LDS in parts
    constexpr int PIECES = HD / 8, ITEMS = PKEYS * PIECES, PER_THREAD = (ITEMS + THREADS - 1) / THREADS;
    constexpr int SETS = HD <= 128 ? 2 : 1;           // steps whose rows wait in registers
    struct Raw { float4 k[PER_THREAD][2], v[PER_THREAD][2]; };
    auto load_kv = [&](int ks, Raw& raw) {
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
            const int item = (tid + i * THREADS) % ITEMS;
            const size_t at = row_address(ks + item / PIECES) + (item % PIECES) * 8;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                raw.k[i][j] = *reinterpret_cast<const float4*>(a.kpool + at + 4 * j);
                raw.v[i][j] = *reinterpret_cast<const float4*>(a.vpool + at + 4 * j);
            }
        }
    };
    auto store_kv = [&](int slot, const Raw& raw) {
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
            const int item = tid + i * THREADS, key = item / PIECES, dim0 = (item % PIECES) * 8;
            const float kv[8] = {raw.k[i][0].x, raw.k[i][0].y, raw.k[i][0].z, raw.k[i][0].w, raw.k[i][1].x, raw.k[i][1].y, raw.k[i][1].z, raw.k[i][1].w};
            const float vv[8] = {raw.v[i][0].x, raw.v[i][0].y, raw.v[i][0].z, raw.v[i][0].w, raw.v[i][1].x, raw.v[i][1].y, raw.v[i][1].z, raw.v[i][1].w};
            const Parts kp = parts8(kv), vp = parts8(vv);
            if (item < ITEMS) {
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    *reinterpret_cast<uint4*>(&lds.k[slot][p][key][dim0]) = kp.p[p];
                    *reinterpret_cast<uint4*>(&lds.v[slot][p][key][dim0]) = vp.p[p];
                }
            }
        }
    };
    auto meet = [] {                                  // (only LDS is ordered here: the loads in flight are not waited for)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    Raw raw[SETS];
    for (int seg0 = 0; seg0 < nsteps;) {
        const int seg_first = kfirst + seg0 * PKEYS;
        lp0 = page_of(max(seg_first, tile_lo));
        const int seg_steps = min(nsteps - seg0, ((lp0 + TBL_MAX) * page_size - seg_first) / PKEYS);
        key_lo = max(seg_first, tile_lo);
        key_hi = min(seg_first + seg_steps * PKEYS, kend) - 1;
        __syncthreads();                   // nobody still reads the previous segment's table or staged tiles
        for (int i = tid; i <= page_of(key_hi) - lp0; i += THREADS) tbl[i] = table[lp0 + i];
        __syncthreads();
        load_kv(seg_first, raw[0]);
        if constexpr (SETS == 2) load_kv(seg_first + PKEYS, raw[1]);
        if constexpr (PSLOTS == 2) {
            store_kv(0, raw[0]);
            load_kv(seg_first + 2 * PKEYS, raw[0]);
        }
        auto step = [&](int s, Raw& next) {
            if (s >= seg_steps) return;
            const int ks = seg_first + s * PKEYS;
            const int slot = PSLOTS == 2 ? (s & 1) : 0;
            meet();                        // with two slots: the step's keys are there; with one: nobody still reads the last step's
            if constexpr (PSLOTS == 1) {
                store_kv(0, next);
                load_kv(ks + SETS * PKEYS, next);
                meet();
            }
            bool act[CB], inner[CB], any_act = false, all_inner = true;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                act[c] = blk_ok[c] && ks <= blk_pmax[c];                                        // else all rows lie before these keys
                inner[c] = act[c] && ks >= blk_lo_max[c] && ks + PKEYS - 1 <= blk_pmin[c];      // every key counts for every row
                any_act = any_act || act[c];
                all_inner = all_inner && inner[c];
            }
            if (any_act) {
                // 1. scores: this lane gets row r of block c, keys ks + 16 * t + 4 * kg + i
                floatx4_t st[CB][2];
#pragma unroll
                for (int c = 0; c < CB; ++c) st[c][0] = st[c][1] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < KC; ++kk) {
                    Parts ka[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int p = 0; p < 3; ++p) {
                            const uint16_t* row = lds.k[slot][p][t * 16 + r];
                            if (kk < KK) {
                                ka[t].p[p] = *reinterpret_cast<const uint4*>(row + kk * 32 + kg * 8);
                            } else {
                                const uint2 half = *reinterpret_cast<const uint2*>(row + KK * 32 + kg * 4);
                                ka[t].p[p] = make_uint4(half.x, half.y, 0u, 0u);
                            }
                        }
#pragma unroll
                    for (int n = 0; n < 6; ++n)
#pragma unroll
                        for (int c = 0; c < CB; ++c)
#pragma unroll
                            for (int t = 0; t < 2; ++t) st[c][t] = times(ka[t].p[PART_A[n]], qf[c][kk].p[PART_B[n]], st[c][t]);
                }
                Parts pf[CB];
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    float sc[8], lane_max = -INFINITY;
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            float v = st[c][t][i];
                            if (!inner[c]) {
                                const int key = ks + t * 16 + kg * 4 + i;
                                v = (row_ok[c] && act[c] && key <= pos[c] && key >= row_lo[c]) ? v : -INFINITY;
                            }
                            sc[t * 4 + i] = v;
                            lane_max = fmaxf(lane_max, v);
                        }
                    // 2. a row whose scores have risen far above its reference: move it, rescale what was summed
                    if (__any(lane_max - REF_SLACK > m_ref[c])) {
                        const float mx = lanes4(lane_max, true);
                        const bool move = mx > m_ref[c] + REF_SLACK;
                        const float m_new = move ? mx : m_ref[c];
                        const float corr = move ? expf(m_ref[c] - m_new) : 1.0f;
                        m_ref[c] = m_new;
                        l_lane[c] *= corr;
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt) o[c][dt] *= corr;
                    }
                    // 3. weights
                    float w[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        w[j] = exp_below(sc[j] - m_ref[c]);
                        l_lane[c] += w[j];
                    }
                    pf[c] = parts8(w);
                }
                // and O^T += V^T . P^T: the A operand of lane (dim r of sixteen, group kg) is V of the keys of the lane's scores
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    uint4 vf[3];
#pragma unroll
                    for (int p = 0; p < 3; ++p) vf[p] = read_v_part(&lds.v[slot][p][0][0], dt * 16, r, kg);
#pragma unroll
                    for (int n = 0; n < 6; ++n)
#pragma unroll
                        for (int c = 0; c < CB; ++c) o[c][dt] = times(vf[PART_A[n]], pf[c].p[PART_B[n]], o[c][dt]);
                }
            }
            if constexpr (PSLOTS == 2) {
                store_kv((s + 1) & 1, next);
                load_kv(ks + 3 * PKEYS, next);
            }
        };
        for (int s0 = 0; s0 < seg_steps; s0 += 2) {
            step(s0, raw[PSLOTS == 2 ? 1 : 0]);
            step(s0 + 1, raw[PSLOTS == 2 || SETS == 1 ? 0 : 1]);
        }
        seg0 += seg_steps;
    }

    float l[CB], zero = 0.f;
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        l[c] = lanes4(l_lane[c], false);
        if (row_ok[c]) {
            zero = fmaf(l[c], 0.f, zero);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int i = 0; i < 4; ++i) zero = fmaf(o[c][dt][i], 0.f, zero);
        }
    }
    if (__syncthreads_or(!(zero == 0.f))) return false;
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        if (!row_ok[c]) continue;
        if (a.nsplit > 1) {
            const size_t p = (static_cast<size_t>(tile.row0 + tt[c]) * a.H + head) * a.nsplit + blockIdx.z;
            if (kg == 0) { a.part_ml[p * 2] = m_ref[c]; a.part_ml[p * 2 + 1] = l[c]; }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<floatx4_t*>(a.part_o + p * HD + dt * 16 + kg * 4) = o[c][dt];
        } else {
            const float inv = 1.0f / l[c];
            float* to = a.out + static_cast<size_t>(tile.row0 + tt[c]) * a.H * HD + static_cast<size_t>(head) * HD + kg * 4;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<floatx4_t*>(to + dt * 16) = o[c][dt] * inv;
        }
    }
    return true;
}

// Blocks of 16 rows a wavefront may own.  A tile has tokens for so many; where they own fewer, two workgroups share it.
constexpr int F32_MAX_BLOCKS = HEAD_DIM <= 64 ? 2 : 1;

template <int CB, bool POW2>
__global__ __launch_bounds__(MA_WAVES * WAVE) __attribute__((amdgpu_waves_per_eu(HEAD_DIM * CB <= 128 ? 2 : 1)))
void mfma_attention_f32_kernel(TileArgs a, const QTile* __restrict__ tiles, int n_tiles) {
    constexpr int HALVES = F32_MAX_BLOCKS / CB;      // workgroups a tile
    union Lds { PartLds parts; ExactLds exact; };
    __shared__ __attribute__((aligned(16))) char lds[sizeof(Lds)];
    __shared__ __attribute__((aligned(16))) int32_t tbl[TBL_MAX];
    // As many workgroups as the chip holds at once; the tiles come sorted by the keys they walk,
    // longest first, and workgroup w takes tiles w, 2P-1-w, 2P+w, ... (P workgroups in x).
    for (int round = 0;; ++round) {
        int tile_at = (round & 1) ? (round + 1) * gridDim.x - 1 - blockIdx.x : round * gridDim.x + blockIdx.x;
        // one round only: a compute unit gets workgroups that stand as many in the grid's order apart as the chip has units;
        // every other such stretch of the grid walks the sorted list backwards, so that long tiles meet short ones there
        const int count = n_tiles * HALVES;
        if (count <= static_cast<int>(gridDim.x) && (blockIdx.y + gridDim.y * blockIdx.z) * gridDim.x / 256 % 2 == 1) tile_at = count - 1 - tile_at;
        if (tile_at >= count || tile_at < 0) break;
        QTile tile = tiles[tile_at / HALVES];
        if constexpr (HALVES == 2) {                 // this workgroup takes one half of the tile's tokens
            const int half = MA_WAVES * (16 >> a.hpt_shift), from = tile_at % 2 * half;
            tile.ntok = min(tile.ntok - from, half);
            if (tile.ntok <= 0) continue;
            tile.row0 += from;
            tile.pos0 += from;
        }
        if (!parts_tile<CB, POW2>(a, tile, *reinterpret_cast<PartLds*>(lds), tbl)) {
#pragma nounroll
            for (int c = 0; c < CB; ++c) {
                __syncthreads();
                exact_tile<POW2>(a, tile, CB, c, *reinterpret_cast<ExactLds*>(lds), tbl);
            }
        }
        __syncthreads();       // the next tile's first stores find nobody reading this one's
    }
}

static int heads_per_tile(int group) { return group >= 16 ? 16 : group > 4 ? 8 : group > 2 ? 4 : group > 1 ? 2 : 1; }

NI_EXPORT int ni_mfma_attention_f32_head_dim() { return HEAD_DIM; }


// Tokens of a tile for `group` query heads per kv head: F32_MAX_BLOCKS blocks of 16 rows for each of four wavefronts.
NI_EXPORT int ni_mfma_attention_f32_tile_tokens(int group) {
    if (group < 1) return 0;
    return MA_WAVES * F32_MAX_BLOCKS * (16 / heads_per_tile(group));
}

// tiles: int32 [n_tiles, 4] rows of (sequence, first row, tokens, first position), at most
// ni_mfma_attention_f32_tile_tokens tokens each, sorted by the keys they walk (longest first).
// part_o: float [T, H, nsplit, HEAD_DIM], part_ml: float [T, H, nsplit, 2]; unused when nsplit == 1.
NI_EXPORT int ni_mfma_attention_f32(const void* q, int q_stride, const void* kpool, const void* vpool,
                                    const void* block_table, int table_stride, const void* tiles, int n_tiles, void* out,
                                    void* part_o, void* part_ml, int H, int KVH, int page_size, int window, float scale,
                                    int nsplit, int blocks, hipStream_t stream) {
    if (n_tiles <= 0) return 0;
    if (H < 1 || KVH < 1 || H % KVH != 0 || page_size < 1 || nsplit < 1 || nsplit > 64 || !(scale > 0.f)) return -1;
    if (nsplit > 1 && (!part_o || !part_ml)) return -2;
    if (q_stride % 4 != 0) return -3;
    const int G = H / KVH;
    const int hpt = heads_per_tile(G);
    int hpt_shift = 0;
    while ((1 << hpt_shift) < hpt) ++hpt_shift;
    const int chunks = (G + hpt - 1) / hpt;
    const bool pow2 = (page_size & (page_size - 1)) == 0;
    int page_shift = 0;
    while (pow2 && (1 << page_shift) < page_size) ++page_shift;
    if (blocks < 1 || blocks > F32_MAX_BLOCKS) return -5;
    const int per_tile = KVH * chunks * nsplit;
    const int count = n_tiles * (F32_MAX_BLOCKS / blocks);      // workgroups' shares of tiles
    auto kernel = pow2 ? mfma_attention_f32_kernel<1, true> : mfma_attention_f32_kernel<1, false>;
    if constexpr (F32_MAX_BLOCKS == 2)
        if (blocks == 2) kernel = pow2 ? mfma_attention_f32_kernel<2, true> : mfma_attention_f32_kernel<2, false>;
    static int slots_of[2][2], units_of[2][2];
    int *slots = slots_of[blocks - 1], *units = units_of[blocks - 1];
    if (slots[pow2] == 0) {
        int dev = 0, cus = 0, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, MA_WAVES * WAVE, 0) != hipSuccess || cus < 1 ||
            per_cu < 1)
            return -4;
        units[pow2] = cus;
        slots[pow2] = cus * per_cu;
    }
    // with no more tiles than the chip holds workgroups every tile gets one (paired over the compute units, see the
    // kernel); else two rounds pair long tiles with short ones, or more, as few as fit the chip
    int rounds = 1;
    if (count * per_tile > slots[pow2]) {
        rounds = 2;
        while ((count + rounds - 1) / rounds * per_tile > slots[pow2] && rounds < count) rounds += 1;
    }
    const int in_x = (count + rounds - 1) / rounds;
    dim3 grid(in_x, KVH * chunks, nsplit);
    const TileArgs args{(const float*)q, (const float*)kpool, (const float*)vpool, (const int32_t*)block_table, (float*)out, (float*)part_o,
                        (float*)part_ml, q_stride, table_stride, H, KVH, page_size, page_shift, hpt_shift, window, nsplit, scale};
    kernel<<<grid, MA_WAVES * WAVE, 0, stream>>>(args, (const QTile*)tiles, n_tiles);
    return NI_LAUNCH_RESULT();
}

// ---------------------------------------------------------------------------------------------
// Single tokens (decode steps, short prompt portions) in true float32: one workgroup per (token,
// kv head, sixteen query heads of its group, run of the key range).  The rows of the products are
// the query heads that share the kv head; the wavefronts of the workgroup take the 16-key steps
// of the run in turn, each with a running (reference, sum, output) of its own, and meet in LDS at
// the end.  Both operands that come from the cache are loaded from global memory straight in the
// layout the matrix instructions want, so nothing is staged and no barrier stands in the loop:
//   K as the A operand of S^T = K . Q^T: lane (r, kg) holds dims kg*HD/4 .. +HD/4 of key r, 64
//     bytes in a row at head size 64 (four lanes read one row between them);
//   V^T as the A operand of O^T += V^T . P^T: for the keys {4*kg + i} of MFMA i, lane (r, kg)
//     holds dims r*HD/16 .. +HD/16 of key 4*kg + i (sixteen lanes read one row between them).
// The rows of a step wait in registers, DEC_DEPTH steps ahead of the arithmetic: two, which leaves the registers
// for two workgroups a compute unit up to head size 128 (with three or four steps ahead a decode batch of mixed
// context lengths ran slower: one workgroup a unit cannot pair a long token with a short one).
#define DEC_WAVES 4
#define DEC_KEYS 16
#define DEC_DEPTH 2

//
// FEW (up to four query heads a kv head, the usual group): rows of a 16 x 16 product past those heads are waste, and a
// step of sixteen keys at head size 128 is 64 instructions of 32 cycles one behind the other on a wavefront that has its
// matrix core to itself.  v_mfma_f32_4x4x1_f32 multiplies sixteen blocks of 4 x 4 in 8 cycles: block (kg, r / 4) is four
// keys or dims by four heads.
//   scores: A lane (r, kg) as above, B the head r % 4 at the same dims; lane (r, kg) gets the keys 4 * (r/4) + i of its head,
//     one quarter of the dims, and the four kg are added up.
//   output: A lane (r, kg) holds dims (4*kg + r%4)*HD/16 .. of key 4 * (r/4) + i, B its own weights; every r / 4 sums its own
//     keys, and they meet at the end.
// Measured, 16 x 16 : 4 x 4, us with the merge: 8 tokens of 774 to 1,300 keys, head size 128, 24 heads on 8, in one / two /
// four runs 39.7 : 33.3, 27.7 : 24.4, 21.8 : 20.5 (68 MB; a run of 325 keys a compute unit is what remains); head size 64, 32 on 8,
// 8 tokens of up to 2,200 keys in two / four runs 24.9 : 21.2, 17.3 : 17.0, 40 tokens of up to 1,300 uncut 37.7 : 34.2.
template <bool POW2, bool FEW>
__global__ __launch_bounds__(DEC_WAVES * WAVE) void mfma_decode_f32_kernel(
    const float* __restrict__ q, int q_stride, const float* __restrict__ kpool, const float* __restrict__ vpool,
    const int32_t* __restrict__ block_table, int table_stride, const int32_t* __restrict__ seq_of_token,
    const int32_t* __restrict__ positions, float* __restrict__ out, float* __restrict__ part_o,
    float* __restrict__ part_ml, int H, int KVH, int page_size, int page_shift, int window, float scale, int nsplit) {
    constexpr int HD = HEAD_DIM;
    constexpr int NW = DEC_WAVES;
    constexpr int THREADS = NW * WAVE;
    constexpr int KS = DEC_KEYS;
    constexpr int QK = HD / 4;                     // MFMAs of the first product per step; floats of Q and of a key a lane holds
    constexpr int DB = HD / 16;                    // MFMAs of the second product per 4 keys
    constexpr int DEPTH = DEC_DEPTH;
    constexpr int ROWS = FEW ? 4 : 16;
    __shared__ __attribute__((aligned(16))) float so[NW][ROWS][HD];      // the wavefronts' outputs, met at the end
    __shared__ float sm_ml[NW][ROWS][2];
    constexpr int TBL_MAX = 1024;
    __shared__ __attribute__((aligned(16))) int32_t tbl[TBL_MAX];

    // (uncut key ranges of many tokens: a compute unit holds workgroups u and u + half the grid, the same x in the
    // lower and the upper half of y; in the order of their contexts the upper half takes the tokens from the far end:
    // a long and a short one on every unit)
    int t = (gridDim.z == 1 && gridDim.y > 1 && 2 * blockIdx.y >= gridDim.y) ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
    if (gridDim.z == 1 && gridDim.y > 1 && gridDim.x > 1 && gridDim.x <= RANKED_TOKENS && gridDim.x * gridDim.y <= RANKED_GROUPS)
        t = token_by_length(positions, gridDim.x, t, tbl);
    const int G = H / KVH;
    const int chunks = (G + 15) / 16;
    const int g = blockIdx.y / chunks;
    const int chunk = blockIdx.y % chunks;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
    const int r = lane % 16, kg = lane / 16;
    const int hh = chunk * 16 + r % ROWS;          // this lane's row: a query head of the group
    const int key4 = 4 * (FEW ? r / 4 : kg);       // first of the lane's four keys of a step
    const int dims = (FEW ? 4 * kg + r % 4 : r) * DB;      // first of the dims it loads of their values
    const bool row_ok = hh < G;
    const int head = g * G + hh;

    const int pos = positions[t];
    const int seq = seq_of_token[t];
    const int hi = pos + 1;
    const int lo = window > 0 ? max(0, hi - window) : 0;
    const int kbeg = lo / KS * KS;
    const int nsteps_all = (hi - kbeg + KS - 1) / KS;
    const int per_split = (nsteps_all + nsplit - 1) / nsplit;
    const int s_begin = blockIdx.z * per_split;
    const int nsteps = max(0, min(nsteps_all, s_begin + per_split) - s_begin);
    const int kfirst = kbeg + s_begin * KS;

    const int32_t* table = block_table + static_cast<size_t>(seq) * table_stride;
    auto page_of = [&](int key) { return POW2 ? (key >> page_shift) : key / page_size; };
    auto slot_of = [&](int key) { return POW2 ? (key & (page_size - 1)) : key % page_size; };
    int key_lo = 0, key_hi = 0, lp0 = 0;
    auto row_address = [&](int key) -> size_t {
        // clamped to keys the token may read: those before `lo` may lie in pages already given back
        const int kc = min(max(key, max(key_lo, lo)), key_hi);
        const int page = tbl[page_of(kc) - lp0];
        return ((static_cast<size_t>(max(page, 0)) * KVH + g) * page_size + slot_of(kc)) * HD;
    };

    // Q, scaled, as the B operand: lane (row r, group kg) holds dims kg*HD/4 .. +HD/4
    float qf[QK];
    if (row_ok) {
        VecIO<float, QK>::load(q + static_cast<size_t>(t) * q_stride + static_cast<size_t>(head) * HD + kg * QK, qf);
#pragma unroll
        for (int j = 0; j < QK; ++j) qf[j] *= scale;
    } else {
#pragma unroll
        for (int j = 0; j < QK; ++j) qf[j] = 0.f;
    }

    float m_ref = NEG_BIG, l_lane = 0.f;       // the row's reference; the sum of this lane's own weights
    floatx4_t o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = floatx4_t{0.f, 0.f, 0.f, 0.f};

    struct StepRows { float k[QK]; float v[4][DB]; };
    auto load_rows = [&](int ks, StepRows& rows) {
        VecIO<float, QK>::load(kpool + row_address(ks + r) + kg * QK, rows.k);
#pragma unroll
        for (int i = 0; i < 4; ++i) VecIO<float, DB>::load(vpool + row_address(ks + key4 + i) + dims, rows.v[i]);
    };

    StepRows ring[DEPTH];
    for (int seg0 = 0; seg0 < nsteps;) {
        key_lo = kfirst + seg0 * KS;
        lp0 = page_of(max(key_lo, lo));
        const int seg_steps = min(nsteps - seg0, ((lp0 + TBL_MAX) * page_size - key_lo) / KS);
        key_hi = min(key_lo + seg_steps * KS, hi) - 1;
        __syncthreads();
        for (int i = tid; i <= page_of(key_hi) - lp0; i += THREADS) tbl[i] = table[lp0 + i];
        __syncthreads();
        // this wavefront's steps of the segment: wave, wave + NW, ...
        const int mine = seg_steps > wave ? (seg_steps - wave + NW - 1) / NW : 0;
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) load_rows(key_lo + (wave + d * NW) * KS, ring[d]);
        // Step j lives in slot j % DEPTH of the ring; the loop is unrolled DEPTH times so that a slot is a
        // fixed set of registers, asked for its next rows as soon as its step has used it.
        auto step = [&](int j, StepRows& rows) {
            const int ks = key_lo + (wave + j * NW) * KS;
            if (j < mine) {
                // 1. scores: this lane gets its row's keys ks + key4 + i
                floatx4_t st = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j1 = 0; j1 < QK; ++j1) {
                    if constexpr (FEW) st = __builtin_amdgcn_mfma_f32_4x4x1f32(rows.k[j1], qf[j1], st, 0, 0, 0);
                    else st = __builtin_amdgcn_mfma_f32_16x16x4f32(rows.k[j1], qf[j1], st, 0, 0, 0);
                }
                if constexpr (FEW) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) st[i] = lanes4(st[i], false);
                }
                const bool inner = ks >= lo && ks + KS - 1 <= pos;
                float sc[4];
                float lane_max = NEG_BIG;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = st[i];
                    if (!inner) {
                        const int key = ks + key4 + i;
                        v = (key <= pos && key >= lo) ? v : NEG_BIG;
                    }
                    sc[i] = v;
                    lane_max = fmaxf(lane_max, v);
                }
                // 2. a row whose scores have risen far above its reference: move it, rescale what was summed
                if (__any(lane_max - REF_SLACK > m_ref)) {
                    const float mx = FEW ? quads4(lane_max, true) : lanes4(lane_max, true);
                    const bool move = mx > 0.5f * NEG_BIG && mx > m_ref + REF_SLACK;
                    const float m_new = move ? mx : m_ref;
                    const float corr = move ? expf(m_ref - m_new) : 1.0f;
                    m_ref = m_new;
                    l_lane *= corr;
#pragma unroll
                    for (int db = 0; db < DB; ++db) o[db] *= corr;
                }
                // 3. weights, and O^T += V^T . P^T for the keys {key4 + i} of MFMA i
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float p = expf(sc[i] - m_ref);
                    if (!inner) p = sc[i] > 0.5f * NEG_BIG ? p : 0.f;
                    l_lane += p;
#pragma unroll
                    for (int db = 0; db < DB; ++db) {
                        if constexpr (FEW) o[db] = __builtin_amdgcn_mfma_f32_4x4x1f32(rows.v[i][db], p, o[db], 0, 0, 0);
                        else o[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(rows.v[i][db], p, o[db], 0, 0, 0);
                    }
                }
            }
            load_rows(ks + DEPTH * NW * KS, rows);
        };
        for (int j0 = 0; j0 < mine; j0 += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) step(j0 + d, ring[d]);
        }
        seg0 += seg_steps;
    }

    // wavefronts meet: every one leaves (reference, sum) of its rows and its 16 x HD output in LDS; this lane
    // holds dims (4*kg + i)*DB + db of its row in o[db][i]
    const float l = FEW ? quads4(l_lane, false) : lanes4(l_lane, false);
    if (kg == 0 && r < ROWS) { sm_ml[wave][r][0] = m_ref; sm_ml[wave][r][1] = l; }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const float v = FEW ? quads4(o[db][i], false) : o[db][i];
            if (r < ROWS) so[wave][r][(4 * kg + i) * DB + db] = v;
        }
    __syncthreads();
    const int rows_here = min(16, G - chunk * 16);
    for (int idx = tid; idx < rows_here * HD; idx += THREADS) {
        const int row = idx / HD, dim = idx % HD;
        float M = sm_ml[0][row][0];
#pragma unroll
        for (int w = 1; w < NW; ++w) M = fmaxf(M, sm_ml[w][row][0]);
        float Lsum = 0.f, O = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float f = expf(sm_ml[w][row][0] - M);
            Lsum += sm_ml[w][row][1] * f;
            O += so[w][row][dim] * f;
        }
        const int h = g * G + chunk * 16 + row;
        if (nsplit == 1) {
            out[static_cast<size_t>(t) * H * HD + static_cast<size_t>(h) * HD + dim] = O / Lsum;
        } else {
            const size_t p = (static_cast<size_t>(t) * H + h) * nsplit + blockIdx.z;
            part_o[p * HD + dim] = O;
            if (dim == 0) { part_ml[p * 2] = M; part_ml[p * 2 + 1] = Lsum; }
        }
    }
}

// Attention of single tokens on the matrix cores in float32: same arguments and partial-result layout as the
// token-at-a-time kernel (`out` is left to its merge kernel when nsplit > 1).
NI_EXPORT int ni_mfma_token_attention_f32(const void* q, int q_stride, const void* kpool, const void* vpool,
                                          const void* block_table, int table_stride, const void* seq_of_token,
                                          const void* positions, void* out, void* part_o, void* part_ml, int T_tokens,
                                          int H, int KVH, int page_size, int window, float scale, int nsplit,
                                          hipStream_t stream) {
    if (T_tokens <= 0) return 0;
    if (H < 1 || KVH < 1 || H % KVH != 0 || page_size < 1 || nsplit < 1 || nsplit > 65535 || !(scale > 0.f)) return -1;
    if (nsplit > 1 && (!part_o || !part_ml)) return -2;
    if (q_stride % 4 != 0) return -3;
    const int G = H / KVH;
    const int chunks = (G + 15) / 16;
    const bool pow2 = (page_size & (page_size - 1)) == 0;
    int page_shift = 0;
    while (pow2 && (1 << page_shift) < page_size) ++page_shift;
    dim3 grid(T_tokens, KVH * chunks, nsplit);
    auto kernel = G <= 4 ? (pow2 ? mfma_decode_f32_kernel<true, true> : mfma_decode_f32_kernel<false, true>)
                         : (pow2 ? mfma_decode_f32_kernel<true, false> : mfma_decode_f32_kernel<false, false>);
    kernel<<<grid, DEC_WAVES * WAVE, 0, stream>>>(
        (const float*)q, q_stride, (const float*)kpool, (const float*)vpool, (const int32_t*)block_table, table_stride,
        (const int32_t*)seq_of_token, (const int32_t*)positions, (float*)out, (float*)part_o, (float*)part_ml, H, KVH,
        page_size, page_shift, window, scale, nsplit);
    return NI_LAUNCH_RESULT();
}
