// Short causal convolutions over time, a filter a channel, for gfx950:
//     y[t, c] = sum_j w[c, j] * u[t - (taps - 1 - j), c]        the last tap is the token's own input
//
// A step brings, for every sequence b, the rows q_start[b] .. q_start[b] + q_len[b] - 1 (consecutive tokens of that
// sequence).  Inputs before a portion's first row come from the sequence's tail, [(taps - 1)][channels] float32 (the
// oldest first; zeros for a new sequence) at float `tail_off` of the row state_slot[b] of `state`.  A step of single
// tokens (`single`: one row a sequence) moves the tail on in the kernel that reads it.  So does a step of one sequence whose first
// taps - 1 rows, the only ones that read the tail, lie in one thread's block of rows (TailMove::Alone); for other portions
// conv_move_tail_kernel does so in a launch of its own, after every row has been read (4.2 to 5.5 us a launch, all latency:
// 2,045 tokens through eight layers with twelve convolutions 3,123 us with it, 3,081 without and with all states cleared in one launch).
//
//   input_conv        x[t] = u[t] + conv(u)[t]: what a sublayer reads of the stream
//   add_norm_conv     h += rmsnorm(y) * w * mult, and (single tokens) the input convolution of the layer behind it
//   qkv_conv          convolution of the projected queries, keys and values, a norm a head, the rotation of neighbouring
//                     channel pairs, and the way into the queries' rows and the cache pages, in one kernel
//
// All arithmetic is float32.  Every entry point returns 0 or a hipError_t.
#include "common.h"

#include <algorithm>
#include <type_traits>

static inline unsigned blocks_of(size_t n, unsigned per) { return static_cast<unsigned>((n + per - 1) / per); }

// where the sequences of a step lie and where their tails are
struct StepRows {
    const int32_t* __restrict__ seq_of_token;
    const int32_t* __restrict__ q_start;
    const int32_t* __restrict__ q_len;
    const int32_t* __restrict__ state_slot;
    float* __restrict__ state;
    size_t state_stride, tail_off;
    __device__ __forceinline__ float* tail(int b) const {
        return state + static_cast<size_t>(state_slot[b]) * state_stride + tail_off;
    }
};

// who moves a sequence's tail on: a launch of its own behind the step's rows, the thread of a single token, or the thread that has the
// first rows of a step's one sequence
enum class TailMove { Behind, Single, Alone };
static TailMove tail_move(bool single, int B, int block, int taps) {
    return single ? TailMove::Single : B == 1 && block >= taps - 1 ? TailMove::Alone : TailMove::Behind;
}

// the filtered input at row t (place r in its portion), channel c of `channels`
__device__ __forceinline__ float conv_at(const float* __restrict__ u, int stride, const float* __restrict__ w, const float* tail,
                                         int t, int r, int c, int channels, int taps) {
    float acc = 0.f;
    for (int j = 0; j < taps; ++j) {
        const int back = taps - 1 - j;            // how many tokens before this one
        const float v = r - back >= 0 ? u[static_cast<size_t>(t - back) * stride + c]
                                      : tail[static_cast<size_t>(taps - 1 + r - back) * channels + c];
        acc += w[static_cast<size_t>(c) * taps + j] * v;
    }
    return acc;
}

// a channel's column of the tail after one more input
__device__ __forceinline__ void move_tail_one(float* tail, int c, int channels, int taps, float input) {
    for (int j = 0; j + 2 < taps; ++j) tail[static_cast<size_t>(j) * channels + c] = tail[static_cast<size_t>(j + 1) * channels + c];
    if (taps > 1) tail[static_cast<size_t>(taps - 2) * channels + c] = input;
}

// N channels' columns of the tail after a portion of n rows that begins at row `first`
template <int N>
__device__ __forceinline__ void move_tail_rows(const float* __restrict__ u, int stride, float* tail, int first, int n, int c, int channels, int taps) {
    const int keep = taps - 1;
    for (int j = 0; j < keep; ++j) {              // ascending: what is read lies at or above what has been written
        const int idx = n - keep + j;             // place in the portion of the input that ends up at j
        float v[N];
        if (idx >= 0) VecIO<float, N>::load(u + static_cast<size_t>(first + idx) * stride + c, v);
        else VecIO<float, N>::load(tail + static_cast<size_t>(keep + idx) * channels + c, v);
        VecIO<float, N>::store(tail + static_cast<size_t>(j) * channels + c, v);
    }
}

// the last taps - 1 inputs of every sequence of the step, the oldest first; a thread moves one channel's column
__global__ void conv_move_tail_kernel(const float* __restrict__ u, int stride, StepRows rows, int channels, int taps, int B) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (c >= channels || b >= B) return;
    const int n = rows.q_len[b];
    if (n > 0) move_tail_rows<1>(u, stride, rows.tail(b), rows.q_start[b], n, c, channels, taps);
}

static void launch_move_tail(const float* u, int stride, const StepRows& rows, int channels, int taps, int B, hipStream_t stream) {
    if (taps < 2) return;
    dim3 grid(blocks_of(channels, 256), B);
    conv_move_tail_kernel<<<grid, 256, 0, stream>>>(u, stride, rows, channels, taps, B);
}

// ---------------------------------------------------------------- x = h + conv(h), in the type of the products
// A thread takes one channel (four neighbouring ones with PIECES) of TOKENS consecutive rows, newest last: a row is read
// once for the thread's tokens, and the rows before them once more.  KEEP: taps - 1 rows stay in registers, at most.
#define INPUT_KEEP 4

template <typename T, bool PIECES, int TOKENS>
__global__ void __launch_bounds__(256)
input_conv_kernel(const float* __restrict__ h, const float* __restrict__ w, StepRows rows, T* __restrict__ x, int Tn, int d, int taps,
                  int per_row, size_t total, TailMove move) {
    constexpr int N = PIECES ? 4 : 1;
    const size_t at = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (at >= total) return;
    const int t0 = static_cast<int>(at / per_row) * TOKENS, c = static_cast<int>(at % per_row) * N;
    const int n_tok = min(TOKENS, Tn - t0);
    float wl[INPUT_KEEP + 1][N];                  // the last taps of the filters, the newest first
#pragma unroll
    for (int k = 0; k <= INPUT_KEEP; ++k)
#pragma unroll
        for (int e = 0; e < N; ++e) wl[k][e] = k < taps ? w[static_cast<size_t>(c + e) * taps + taps - 1 - k] : 0.f;
    float own[TOKENS][N];
#pragma unroll
    for (int tt = 0; tt < TOKENS; ++tt)
        if (tt < n_tok) VecIO<float, N>::load(h + static_cast<size_t>(t0 + tt) * d + c, own[tt]);
#pragma unroll
    for (int tt = 0; tt < TOKENS; ++tt) {
        if (tt >= n_tok) break;
        const int t = t0 + tt, b = rows.seq_of_token[t], r = t - rows.q_start[b];
        float* tail = rows.tail(b);
        float acc[N];
#pragma unroll
        for (int e = 0; e < N; ++e) acc[e] = own[tt][e] + wl[0][e] * own[tt][e];
        // the row `back` tokens before this one: the thread's own, another of the step, or of the tail
        auto before = [&](int back, float (&v)[N]) {
            VecIO<float, N>::load(r - back >= 0 ? h + static_cast<size_t>(t - back) * d + c
                                                : tail + static_cast<size_t>(taps - 1 + r - back) * d + c, v);
        };
#pragma unroll
        for (int back = 1; back <= INPUT_KEEP; ++back) {
            if (back >= taps) break;
            float v[N];
            if (back <= tt && r - back >= 0) {
#pragma unroll
                for (int e = 0; e < N; ++e) v[e] = own[tt >= back ? tt - back : 0][e];
            } else {
                before(back, v);
            }
#pragma unroll
            for (int e = 0; e < N; ++e) acc[e] += wl[back][e] * v[e];
        }
        for (int back = INPUT_KEEP + 1; back < taps; ++back) {
            float v[N];
            before(back, v);
#pragma unroll
            for (int e = 0; e < N; ++e) acc[e] += w[static_cast<size_t>(c + e) * taps + taps - 1 - back] * v[e];
        }
        if constexpr (PIECES) store_packed<T, 4>(x + static_cast<size_t>(t) * d + c, acc);
        else st(x + static_cast<size_t>(t) * d + c, acc[0]);
        if (move == TailMove::Single) {        // this thread alone reads and writes its channels' columns of the tail
#pragma unroll
            for (int e = 0; e < N; ++e) move_tail_one(tail, c + e, d, taps, own[tt][e]);
        }
    }
    if (move == TailMove::Alone && t0 == 0) move_tail_rows<N>(h, d, rows.tail(0), rows.q_start[0], rows.q_len[0], c, d, taps);      // (as above)
}

static bool whole_pieces(int d, const StepRows& rows, const void* a, const void* b) {
    return d % 4 == 0 && rows.state_stride % 4 == 0 && rows.tail_off % 4 == 0 && reinterpret_cast<uintptr_t>(rows.state) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(a) % 16 == 0 && reinterpret_cast<uintptr_t>(b) % 16 == 0;
}

// h float32 [T, d], w float32 [d, taps], x [T, d] of the type `dtype` (0 float32, 1 bfloat16)
NI_EXPORT int ni_input_conv(const void* h, const void* w, void* state, size_t state_stride, size_t tail_off, const void* seq_of_token,
                            const void* q_start, const void* q_len, const void* state_slot, void* x, int T, int B, int d, int taps,
                            int single, int dtype, hipStream_t stream) {
    const size_t total = static_cast<size_t>(T) * d;
    if (total == 0 || B <= 0) return 0;
    if (taps < 1 || state_stride < tail_off + static_cast<size_t>(taps - 1) * d || (single && T != B)) return -1;
    const StepRows rows{(const int32_t*)seq_of_token, (const int32_t*)q_start, (const int32_t*)q_len, (const int32_t*)state_slot,
                        (float*)state, state_stride, tail_off};
    const bool pieces = whole_pieces(d, rows, h, x);
    const int per_row = pieces ? d / 4 : d;
    TailMove move = TailMove::Behind;
    auto launch = [&](auto* out, auto piece_tag, auto tokens_tag) {
        constexpr int TOKENS = decltype(tokens_tag)::value;
        const size_t threads = static_cast<size_t>((T + TOKENS - 1) / TOKENS) * per_row;
        input_conv_kernel<std::remove_pointer_t<decltype(out)>, decltype(piece_tag)::value, TOKENS><<<blocks_of(threads, 256), 256, 0, stream>>>(
            (const float*)h, (const float*)w, rows, out, T, d, taps, per_row, threads, move = tail_move(single != 0, B, TOKENS, taps));
    };
    auto run = [&](auto* out) {
        using One = std::integral_constant<int, 1>;
        using Four = std::integral_constant<int, 4>;
        // (one sequence in blocks of four from 64 rows on where that moves its tail: the fewer threads cost less than the launch behind them.  100 / 200 rows of
        // 2,048 channels, four taps 6.7 -> 6.2 us, 8.5 -> 6.2; with seven, whose tail takes that launch, blocks of four are 11.5 and 11.6 for 8.0 and 10.0)
        if (pieces) T >= 256 || (T >= 64 && tail_move(single != 0, B, 4, taps) == TailMove::Alone) ? launch(out, std::true_type{}, Four{}) : launch(out, std::true_type{}, One{});
        else launch(out, std::false_type{}, One{});
    };
    if (dtype == 0) run((float*)x);
    else run((bf16_t*)x);
    if (move == TailMove::Behind) launch_move_tail((const float*)h, d, rows, d, taps, B, stream);
    return NI_LAUNCH_RESULT();
}

// ---------------------------------------------------------------- h += rmsnorm(sum of addends) * w * mult, then what reads it
// One workgroup a token, its row in registers between the sum of squares and the division.  x, if given: the new
// stream in the type of the products, or (CONV, steps of single tokens) the new stream plus its convolution for the
// layer behind, whose tail is moved on.
#define NORM_ITEMS 8            // elements of a row a thread keeps: rows of up to 8 * 1024 elements

template <typename X, bool CONV, int VEC>
__global__ void __launch_bounds__(1024)
add_norm_kernel(float* __restrict__ h, const float* __restrict__ addends, int n_addends, size_t addend_stride, const float* __restrict__ w,
                float mult, float eps, X* __restrict__ x, int d, const float* __restrict__ filters, int taps, StepRows rows) {
    constexpr int PIECES = NORM_ITEMS / VEC;      // of VEC neighbouring elements each
    __shared__ float scratch[16];
    const int t = blockIdx.x;
    const size_t base = static_cast<size_t>(t) * d;
    float* tail = nullptr;
    if constexpr (CONV) tail = rows.tail(rows.seq_of_token[t]);
    // everything that does not wait for the sum of squares is read before it
    float y[PIECES][VEC], hv[PIECES][VEC], wn[PIECES][VEC], past[PIECES][VEC], now[PIECES][VEC];
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
        const int i = (threadIdx.x + u * blockDim.x) * VEC;
        if (i < d) {
            VecIO<float, VEC>::load(addends + base + i, y[u]);
            for (int s = 1; s < n_addends; ++s) {
                float a[VEC];
                VecIO<float, VEC>::load(addends + s * addend_stride + base + i, a);
#pragma unroll
                for (int e = 0; e < VEC; ++e) y[u][e] += a[e];
            }
            VecIO<float, VEC>::load(h + base + i, hv[u]);
            VecIO<float, VEC>::load(w + i, wn[u]);
            if constexpr (CONV) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    past[u][e] = 0.f;
                    now[u][e] = filters[static_cast<size_t>(i + e) * taps + taps - 1];
                }
                for (int j = 0; j + 1 < taps; ++j) {
                    float v[VEC];
                    VecIO<float, VEC>::load(tail + static_cast<size_t>(j) * d + i, v);
#pragma unroll
                    for (int e = 0; e < VEC; ++e) past[u][e] += filters[static_cast<size_t>(i + e) * taps + j] * v[e];
                    if (j > 0) VecIO<float, VEC>::store(tail + static_cast<size_t>(j - 1) * d + i, v);
                }
            }
#pragma unroll
            for (int e = 0; e < VEC; ++e) ss += y[u][e] * y[u][e];
        }
    }
    const float inv = 1.0f / sqrtf(block_sum(ss, scratch) / static_cast<float>(d) + eps);
#pragma unroll
    for (int u = 0; u < PIECES; ++u) {
        const int i = (threadIdx.x + u * blockDim.x) * VEC;
        if (i < d) {
            float v[VEC], out[VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                v[e] = hv[u][e] + mult * ((y[u][e] * inv) * wn[u][e]);
                out[e] = v[e];
                if constexpr (CONV) out[e] = (v[e] + past[u][e]) + now[u][e] * v[e];
            }
            VecIO<float, VEC>::store(h + base + i, v);
            if constexpr (CONV) {
                if (taps > 1) VecIO<float, VEC>::store(tail + static_cast<size_t>(taps - 2) * d + i, v);
            }
            if (x) {
                if constexpr (VEC == 4) store_packed<X, 4>(x + base + i, out);
                else st(x + base + i, out[0]);
            }
        }
    }
}

// the same for rows of more elements than the registers take
template <typename X>
__global__ void __launch_bounds__(1024)
add_norm_long_kernel(float* __restrict__ h, const float* __restrict__ addends, int n_addends, size_t addend_stride,
                     const float* __restrict__ w, float mult, float eps, X* __restrict__ x, int d) {
    __shared__ float scratch[16];
    const size_t base = static_cast<size_t>(blockIdx.x) * d;
    auto sum_at = [&](int i) -> float {
        float a = addends[base + i];
        for (int s = 1; s < n_addends; ++s) a += addends[s * addend_stride + base + i];
        return a;
    };
    float ss = 0.f;
    for (int i = threadIdx.x; i < d; i += blockDim.x) {
        const float a = sum_at(i);
        ss += a * a;
    }
    const float inv = 1.0f / sqrtf(block_sum(ss, scratch) / static_cast<float>(d) + eps);
    for (int i = threadIdx.x; i < d; i += blockDim.x) {
        const float v = h[base + i] + mult * ((sum_at(i) * inv) * w[i]);
        h[base + i] = v;
        if (x) st(x + base + i, v);
    }
}

NI_EXPORT int ni_add_norm_max() { return NORM_ITEMS * 1024; }

// addends float32 [n_addends][T][d] (summed in their order), w float32 [d].  filters (float32 [d, taps], or null): x is
// the new stream plus its convolution; a step of single tokens (T == B) only, d at most ni_add_norm_max().
NI_EXPORT int ni_add_norm(void* h, const void* addends, int n_addends, const void* w, float mult, float eps, void* x, int x_dtype, int T,
                          int d, const void* filters, int taps, void* state, size_t state_stride, size_t tail_off,
                          const void* seq_of_token, const void* state_slot, int B, hipStream_t stream) {
    if (T <= 0 || d <= 0) return 0;
    if (n_addends < 1 || !addends) return -1;
    const size_t stride = static_cast<size_t>(T) * d;
    const StepRows rows{(const int32_t*)seq_of_token, nullptr, nullptr, (const int32_t*)state_slot, (float*)state, state_stride, tail_off};
    if (filters && (taps < 1 || !x || T != B || d > NORM_ITEMS * 1024 || state_stride < tail_off + static_cast<size_t>(taps - 1) * d)) return -1;
    if (d > NORM_ITEMS * 1024) {
        auto run_long = [&](auto* out) {
            add_norm_long_kernel<std::remove_pointer_t<decltype(out)>><<<T, 1024, 0, stream>>>((float*)h, (const float*)addends, n_addends, stride,
                                                                                               (const float*)w, mult, eps, out, d);
        };
        if (x_dtype == 0) run_long((float*)x);
        else run_long((bf16_t*)x);
        return NI_LAUNCH_RESULT();
    }
    const bool pieces = d % 4 == 0 && reinterpret_cast<uintptr_t>(h) % 16 == 0 && reinterpret_cast<uintptr_t>(addends) % 16 == 0 &&
                        reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                        (!filters || (state_stride % 4 == 0 && tail_off % 4 == 0 && reinterpret_cast<uintptr_t>(state) % 16 == 0));
    // one piece a thread (few rows: as many threads as there are elements), a whole row at most a workgroup
    const int items = pieces ? d / 4 : d;
    const int threads = std::min(1024, std::max(64, (items + WAVE - 1) / WAVE * WAVE));
    auto run = [&](auto* out) {
        using X = std::remove_pointer_t<decltype(out)>;
        auto go = [&](auto conv_tag, auto vec_tag) {
            add_norm_kernel<X, decltype(conv_tag)::value, decltype(vec_tag)::value><<<T, threads, 0, stream>>>(
                (float*)h, (const float*)addends, n_addends, stride, (const float*)w, mult, eps, out, d, (const float*)filters, taps, rows);
        };
        using One = std::integral_constant<int, 1>;
        using Four = std::integral_constant<int, 4>;
        if (filters) pieces ? go(std::true_type{}, Four{}) : go(std::true_type{}, One{});
        else pieces ? go(std::false_type{}, Four{}) : go(std::false_type{}, One{});
    };
    if (x_dtype == 0) run((float*)x);
    else run((bf16_t*)x);
    return NI_LAUNCH_RESULT();
}

// ---------------------------------------------------------------- projected queries, keys and values on their way to attention
// proj float32 [T, row_stride] holds q [H][maps][dk] | k [G][maps][dk] | v [G][dv] as projected (a head has `maps` query
// and key vectors: attention that combines several maps over the same values).  Every channel is convolved over time
// (filters null: not), every query and key vector is divided by its root mean square and multiplied by a weight [dk]
// shared by all of them (null: not), then its first `rot` channels are rotated, channel 2p with channel 2p + 1, by
// position * freq[p].  Queries go to q_out [T][G][maps][H / G][dk] in the type of the products (the heads of a key head
// and map together), keys to kpool [page][G][slot][maps * dk], values to vpool [page][G][slot][dv].
//
// A wavefront takes UPW units (a query vector, a key vector, or up to a unit's width of a value) of TB consecutive rows, a
// lane two neighbouring channels of every 128; the rows a token needs of its predecessors stay in registers (TAPS > 0) or
// are read again.  The angles of the block's rows are worked out once for all units.
struct QkvForm {
    int H, G, maps, dk, dv, rot, taps, page_size;
};
#define CONV_PAIRS 256          // rotated pairs of a head at most

// two neighbouring elements (PAIRS: sizes and rows are even, the address is aligned to both)
template <bool PAIRS>
__device__ __forceinline__ void load_two(const float* p, const bool (&in)[2], float (&v)[2]) {
    if constexpr (PAIRS) {
        float2 a = make_float2(0.f, 0.f);
        if (in[0]) a = *reinterpret_cast<const float2*>(p);
        v[0] = a.x;
        v[1] = a.y;
    } else {
        v[0] = in[0] ? p[0] : 0.f;
        v[1] = in[1] ? p[1] : 0.f;
    }
}

template <bool PAIRS, typename T>
__device__ __forceinline__ void store_two(T* p, const bool (&in)[2], float a, float b) {
    if constexpr (PAIRS) {
        if (!in[0]) return;
        if constexpr (sizeof(T) == 2) *reinterpret_cast<uint32_t*>(p) = pack_bf16x2(a, b);
        else *reinterpret_cast<float2*>(p) = make_float2(a, b);
    } else {
        if (in[0]) st(p, a);
        if (in[1]) st(p + 1, b);
    }
}

// the sum over the 64 / UPW neighbouring lanes of a unit, every one of them gets it: inside a row of sixteen by
// data-parallel moves, across rows by the swaps of gfx950; no trip through the LDS crossbar
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int UPW> __device__ __forceinline__ float unit_sum(float v) {
    v += dpp_move<0xB1>(v);       // quad_perm [1, 0, 3, 2]
    v += dpp_move<0x4E>(v);       // quad_perm [2, 3, 0, 1]
    v += dpp_move<0x141>(v);      // row_half_mirror: lane i <-> 7 - i of its eight
    v += dpp_move<0x140>(v);      // row_mirror: lane i <-> 15 - i of its sixteen
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    if constexpr (UPW == 1) {
        const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
    }
    return v;
}

template <typename T, int TAPS, int TB, int NP, int UPW, bool PAIRS>
__global__ void __launch_bounds__(256)
qkv_conv_kernel(const float* __restrict__ proj, int row_stride, const int32_t* __restrict__ positions,
                const int32_t* __restrict__ slot_mapping, const float* __restrict__ filters, const float* __restrict__ wq,
                const float* __restrict__ wk, float eps, const float* __restrict__ freq, StepRows rows, T* __restrict__ q_out,
                T* __restrict__ kpool, T* __restrict__ vpool, int Tn, QkvForm f, TailMove move) {
    static_assert(UPW == 1 || NP == 1, "a unit of two a wavefront has one pair a lane");
    __shared__ float cos_of[TB * CONV_PAIRS], sin_of[TB * CONV_PAIRS];
    const int t0 = blockIdx.x * TB, n_tok = min(TB, Tn - t0);
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
    constexpr int GROUP = WAVE / UPW, WIDE = 2 * GROUP * NP;           // lanes of a unit; channels of a unit at most
    const int sub = lane % GROUP;
    const int pairs = f.rot / 2;
    for (int e = tid; e < n_tok * pairs; e += blockDim.x) {
        const int tt = e / pairs, p = e % pairs;
        float sn, cs;
        sincosf(static_cast<float>(positions[t0 + tt]) * freq[p], &sn, &cs);
        cos_of[tt * pairs + p] = cs;
        sin_of[tt * pairs + p] = sn;
    }
    if (pairs) __syncthreads();
    const int nq = f.H * f.maps, nk = f.G * f.maps;
    const int v_parts = (f.dv + WIDE - 1) / WIDE;                      // a value needs no norm: a long one is several units
    const int units = nq + nk + f.G * v_parts;
    const int channels = nq * f.dk + nk * f.dk + f.G * f.dv;
    const int group = f.H / f.G;
    constexpr int KEEP = TAPS > 1 ? TAPS - 1 : 1;
    const int taps = TAPS > 0 ? TAPS : f.taps;
    const int step = gridDim.y * (blockDim.x / WAVE) * UPW;
    for (int first = (blockIdx.y * (blockDim.x / WAVE) + wave) * UPW; first < units; first += step) {
        const int unit = min(first + lane / GROUP, units - 1);         // (a group of lanes without a unit repeats the last one, and stores nothing)
        const bool mine = first + lane / GROUP < units;
        const bool is_q = unit < nq, is_v = unit >= nq + nk;
        const int v_head = is_v ? (unit - nq - nk) / v_parts : 0, v_at = is_v ? (unit - nq - nk) % v_parts * WIDE : 0;
        const int size = is_v ? min(f.dv - v_at, WIDE) : f.dk;
        const int c0 = is_v ? (nq + nk) * f.dk + v_head * f.dv + v_at : unit * f.dk;      // first channel of the unit
        const float* weight = is_v ? nullptr : (is_q ? wq : wk);
        float wt[NP][2][TAPS > 0 ? TAPS : 1], win[NP][2][KEEP];
        bool in[NP][2];
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int c = 2 * sub + 128 * p + e;
                in[p][e] = mine && c < size;
                if constexpr (TAPS == 4) {        // a channel's taps are one 16-byte piece
                    const float4 f4 = in[p][e] ? *reinterpret_cast<const float4*>(filters + static_cast<size_t>(c0 + c) * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
                    wt[p][e][0] = f4.x; wt[p][e][1] = f4.y; wt[p][e][2] = f4.z; wt[p][e][3] = f4.w;
                } else if constexpr (TAPS > 0) {
#pragma unroll
                    for (int j = 0; j < TAPS; ++j) wt[p][e][j] = in[p][e] ? filters[static_cast<size_t>(c0 + c) * TAPS + j] : 0.f;
                }
            }
        float y[TB][NP][2];                       // the block's rows, asked for together; then what becomes of them
#pragma unroll
        for (int tt = 0; tt < TB; ++tt)
#pragma unroll
            for (int p = 0; p < NP; ++p)          // (past the step's end the last row again: no load is under a branch of the block's)
                load_two<PAIRS>(proj + static_cast<size_t>(t0 + min(tt, n_tok - 1)) * row_stride + c0 + 2 * sub + 128 * p, in[p], y[tt][p]);
        // the convolution, from the newest tap back
#pragma unroll
        for (int tt = 0; tt < TB; ++tt) {
            if (tt >= n_tok) break;
            const int t = t0 + tt;
            const int b = rows.seq_of_token[t];
            const int r = t - rows.q_start[b];
            float* tail = filters ? rows.tail(b) : nullptr;
            if constexpr (TAPS > 0) {
                if (tt == 0 || r == 0) {          // the same for the whole wavefront: the rows before this block's or portion's first
                    const float* row = proj + static_cast<size_t>(t) * row_stride + c0;
#pragma unroll
                    for (int j = 0; j < TAPS - 1; ++j) {
                        const int back = TAPS - 1 - j;
                        const float* from = r - back >= 0 ? row - static_cast<ptrdiff_t>(back) * row_stride
                                                          : tail + static_cast<size_t>(TAPS - 1 + r - back) * channels + c0;
#pragma unroll
                        for (int p = 0; p < NP; ++p) {
                            float v[2];
                            load_two<PAIRS>(from + 2 * sub + 128 * p, in[p], v);
                            win[p][0][j] = v[0];
                            win[p][1][j] = v[1];
                        }
                    }
                }
            }
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const int c = 2 * sub + 128 * p;
                const float own[2] = {y[tt][p][0], y[tt][p][1]};
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    if constexpr (TAPS > 0) {
                        float acc = 0.f;
#pragma unroll
                        for (int j = 0; j < TAPS - 1; ++j) acc += wt[p][e][j] * win[p][e][j];
                        y[tt][p][e] = acc + wt[p][e][TAPS - 1] * own[e];
#pragma unroll
                        for (int j = 0; j + 1 < TAPS - 1; ++j) win[p][e][j] = win[p][e][j + 1];
                        if constexpr (TAPS > 1) win[p][e][TAPS - 2] = own[e];
                    } else if (filters) {
                        y[tt][p][e] = in[p][e] ? conv_at(proj, row_stride, filters, tail, t, r, c0 + c + e, channels, taps) : 0.f;
                    }
                }
                if (move == TailMove::Single && filters) {          // this lane alone reads and writes its channels' columns of the tail
                    if constexpr (TAPS > 1) {     // the window holds what the tail is to hold
#pragma unroll
                        for (int j = 0; j < TAPS - 1; ++j)
                            store_two<PAIRS>(tail + static_cast<size_t>(j) * channels + c0 + c, in[p], win[p][0][j], win[p][1][j]);
                    } else {
                        if (in[p][0]) move_tail_one(tail, c0 + c, channels, taps, own[0]);
                        if (in[p][1]) move_tail_one(tail, c0 + c + 1, channels, taps, own[1]);
                    }
                }
            }
        }
        if constexpr (TAPS > 1 && TB >= TAPS - 1) {
            if (move == TailMove::Alone && t0 == 0 && filters) {          // (as above: the only rows that read the tail are this block's)
                float* tail = rows.tail(0);
                const int end = rows.q_start[0] + rows.q_len[0], keep = min(TAPS - 1, rows.q_len[0]);
#pragma unroll
                for (int j = 0; j < TAPS - 1; ++j) {                      // (ascending: what is read lies above what has been written)
                    const float* from = j >= TAPS - 1 - keep ? proj + static_cast<size_t>(end - (TAPS - 1) + j) * row_stride
                                                             : tail + static_cast<size_t>(j + keep) * channels;
#pragma unroll
                    for (int p = 0; p < NP; ++p) {
                        float v[2];
                        load_two<PAIRS>(from + c0 + 2 * sub + 128 * p, in[p], v);
                        store_two<PAIRS>(tail + static_cast<size_t>(j) * channels + c0 + 2 * sub + 128 * p, in[p], v[0], v[1]);
                    }
                }
            }
        }
        // the norm, the block's sums side by side (values and vectors without a weight pass)
        float nw[NP][2];
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int e = 0; e < 2; ++e) nw[p][e] = in[p][e] && weight ? weight[2 * sub + 128 * p + e] : 1.f;
#pragma unroll
        for (int tt = 0; tt < TB; ++tt) {
            float ss = 0.f;
#pragma unroll
            for (int p = 0; p < NP; ++p) ss += y[tt][p][0] * y[tt][p][0] + y[tt][p][1] * y[tt][p][1];
            ss = unit_sum<UPW>(ss);
            const float inv = weight ? 1.0f / sqrtf(ss / static_cast<float>(size) + eps) : 1.f;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                y[tt][p][0] = (y[tt][p][0] * inv) * nw[p][0];
                y[tt][p][1] = (y[tt][p][1] * inv) * nw[p][1];
            }
        }
        // the rotation and the way out
        const int map = is_q ? unit % f.maps : (unit - nq) % f.maps, hd = is_q ? unit / f.maps : 0, g = is_q ? 0 : is_v ? v_head : (unit - nq) / f.maps;
        const size_t q_at = static_cast<size_t>((hd / group) * f.maps + map) * group + hd % group;
#pragma unroll
        for (int tt = 0; tt < TB; ++tt) {
            if (tt >= n_tok) break;
            const int t = t0 + tt;
            const int slot = slot_mapping[t];
            T* dst = nullptr;
            if (is_q) {
                dst = q_out + (static_cast<size_t>(t) * nq + q_at) * f.dk;
            } else if (slot >= 0) {
                const size_t page = slot / f.page_size, in_page = slot % f.page_size, at = (page * f.G + g) * f.page_size + in_page;
                dst = is_v ? vpool + at * f.dv + v_at : kpool + at * (f.maps * f.dk) + map * f.dk;
            }
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const int c = 2 * sub + 128 * p;
                float a = y[tt][p][0], z = y[tt][p][1];
                if (!is_v && c < f.rot) {         // rot is even: both channels of the pair turn
                    const float cs = cos_of[tt * pairs + c / 2], sn = sin_of[tt * pairs + c / 2];
                    const float u = a;
                    a = u * cs - z * sn;
                    z = z * cs + u * sn;
                }
                if (dst) store_two<PAIRS>(dst + c, in[p], a, z);
            }
        }
    }
}

struct QkvArgs {
    const float* proj; int row_stride; const int32_t *positions, *slot_mapping; const float *filters, *wq, *wk; float eps;
    const float* freq; StepRows rows; void *q_out, *kpool, *vpool; int T, B; QkvForm f; bool single;
};

template <typename T, int TAPS, int TB>
static bool launch_qkv(const QkvArgs& a, TailMove& move, hipStream_t stream) {
    move = tail_move(a.single, a.B, TAPS > 1 ? TB : 0, a.f.taps);      // (without a number of taps of its own the kernel has no block)
    const int blocks = (a.T + TB - 1) / TB;
    // every row, unit and tail starts at an even element, and the addresses are aligned to pairs
    auto even = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 8 == 0; };
    const bool pairs = a.f.dk % 2 == 0 && a.f.dv % 2 == 0 && a.row_stride % 2 == 0 && even(a.proj) && even(a.q_out) && even(a.kpool) &&
                       even(a.vpool) && (!a.filters || (even(a.rows.state) && a.rows.state_stride % 2 == 0 && a.rows.tail_off % 2 == 0));
    auto go = [&](auto np, auto upw, auto pair_tag) {
        constexpr int NP = decltype(np)::value, UPW = decltype(upw)::value, WIDE = 128 * NP / UPW;
        const int units = (a.f.H + a.f.G) * a.f.maps + a.f.G * ((a.f.dv + WIDE - 1) / WIDE);
        // as many units a wavefront at once as it takes, several in turn where that leaves the chip full (the block's angles
        // are worked out once for all of them)
        const int most = (units + 4 * UPW - 1) / (4 * UPW);
        const dim3 grid(blocks, std::max(1, std::min(most, (1536 + blocks - 1) / blocks)));
        qkv_conv_kernel<T, TAPS, TB, NP, UPW, decltype(pair_tag)::value><<<grid, 256, 0, stream>>>(
            a.proj, a.row_stride, a.positions, a.slot_mapping, a.filters, a.wq, a.wk, a.eps, a.freq, a.rows, (T*)a.q_out, (T*)a.kpool,
            (T*)a.vpool, a.T, a.f, move);
    };
    auto run = [&](auto np, auto upw) {
        if (pairs) { go(np, upw, std::true_type{}); return true; }
        if constexpr (TAPS == 0) { go(np, upw, std::false_type{}); return true; }
        return false;                             // (a number of taps of its own goes with pairs only)
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    if (a.f.dk <= 64) return run(One{}, Two{});
    if (a.f.dk <= 128) return run(One{}, One{});
    if (TAPS > 0 && a.f.dk <= 256) return run(Two{}, One{});
    return run(std::integral_constant<int, 4>{}, One{});
}

template <typename T>
static TailMove launch_qkv_any(const QkvArgs& a, hipStream_t stream) {
    const bool few = a.T < 64;        // few tokens: a row a workgroup, spread over the units
    TailMove move;
    if (a.filters && a.f.taps == 4 && reinterpret_cast<uintptr_t>(a.filters) % 16 == 0 &&
        (few ? launch_qkv<T, 4, 1>(a, move, stream) : launch_qkv<T, 4, 8>(a, move, stream))) return move;
    few ? launch_qkv<T, 0, 1>(a, move, stream) : launch_qkv<T, 0, 8>(a, move, stream);
    return move;
}

// filters float32 [channels, taps] or null; state and tail_off: see StepRows (channels of the tail: q | k | v)
NI_EXPORT int ni_qkv_conv(const void* proj, int row_stride, const void* positions, const void* slot_mapping, const void* filters, int taps,
                          const void* wq, const void* wk, float eps, const void* freq, int rot, void* state, size_t state_stride,
                          size_t tail_off, const void* seq_of_token, const void* q_start, const void* q_len, const void* state_slot,
                          void* q_out, void* kpool, void* vpool, int T, int B, int H, int G, int maps, int dk, int dv, int page_size,
                          int single, int dtype, hipStream_t stream) {
    if (T <= 0 || B <= 0) return 0;
    if (H < 1 || G < 1 || H % G || maps < 1 || dk < 1 || dv < 1 || dk > 512 || dv > 512 || page_size < 1) return -1;
    const int channels = (H + G) * maps * dk + G * dv;
    if (row_stride < channels || rot < 0 || rot % 2 || rot > dk || rot > 2 * CONV_PAIRS || (rot && !freq)) return -1;
    if (filters && (taps < 1 || state_stride < tail_off + static_cast<size_t>(taps - 1) * channels)) return -1;
    if (single && T != B) return -1;
    const StepRows rows{(const int32_t*)seq_of_token, (const int32_t*)q_start, (const int32_t*)q_len, (const int32_t*)state_slot,
                        (float*)state, state_stride, tail_off};
    const QkvArgs a{(const float*)proj, row_stride, (const int32_t*)positions, (const int32_t*)slot_mapping, (const float*)filters,
                    (const float*)wq, (const float*)wk, eps, (const float*)freq, rows, q_out, kpool, vpool, T, B,
                    QkvForm{H, G, maps, dk, dv, rot, taps, page_size}, single != 0};
    const TailMove move = dtype == 0 ? launch_qkv_any<float>(a, stream) : launch_qkv_any<bf16_t>(a, stream);
    if (filters && move == TailMove::Behind) launch_move_tail((const float*)proj, row_stride, rows, channels, taps, B, stream);
    return NI_LAUNCH_RESULT();
}
