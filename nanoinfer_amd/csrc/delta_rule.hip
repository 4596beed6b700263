// The gated delta rule with one decay per key channel, for gfx950.
//
// Per head, with S [key channel, value channel] float32 carried from token to token:
//     S <- diag(g_t) S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
// Six kernels:
//   delta_prepare      per token, in parallel: the short causal convolutions of q, k, v with silu, the unit
//                      norms of q and k, beta = sigmoid, g = exp(-exp(A) softplus(z + dt)), the output gate
//   conv_state_update  per sequence: the last taps - 1 inputs of the convolutions, kept for the next step
//   delta_rule         per (sequence, head, group of value channels): the recurrence over the step's tokens
//   headnorm_gate      o / rms(o) * w * gate per head, rounded to the compute type for the output product
//   delta_chunk_prepare, delta_chunk_scan   the same recurrence for portions of prompts, sixteen tokens at a
//                      time on the matrix cores (described above them)
//
// The columns of S are independent of one another: u_t[j] and o_t[j] need column j alone.  A column is
// held by PARTS neighbouring lanes, KPT key channels each, in registers for the whole step; the three
// dot products of a token (S^T k, S^T q, k . q) are finished with PARTS-wide butterflies, and one pass
// over the registers serves both the decay and the dot products, because
//     o_t = (gS)^T q + u_t (k . q).
// The state is stored transposed, [head, value channel, key channel], so that the lanes of a column
// read and write neighbouring pieces.  Compiled per (KPT, PARTS); the key size is KPT * PARTS.
#include "common.h"

#include <algorithm>

#ifndef KPT
#define KPT 4
#endif
#ifndef PARTS
#define PARTS 16
#endif

// Sum over the PARTS neighbouring lanes that hold one column (PARTS a power of two up to 16, aligned: they lie in
// one row of sixteen lanes), every lane getting the total, by data-parallel moves inside the row: pairs, quads, the
// mirrored half, the mirrored row.  No trip through the LDS crossbar stands in the recurrence's chain.
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int N> __device__ __forceinline__ float parts_sum(float v) {
    if constexpr (N >= 2) v += dpp_move<0xB1>(v);       // quad_perm [1, 0, 3, 2]
    if constexpr (N >= 4) v += dpp_move<0x4E>(v);       // quad_perm [2, 3, 0, 1]
    if constexpr (N >= 8) v += dpp_move<0x141>(v);      // row_half_mirror: lane i <-> 7 - i of its eight
    if constexpr (N >= 16) v += dpp_move<0x140>(v);     // row_mirror: lane i <-> 15 - i of its sixteen
    return v;
}

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float silu_f(float z) { return z * sigmoid_f(z); }
__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// proj float32 [T, proj_cols]: q [G*dk] | k [G*dk] | v [H*dv] | b [H] as projected.
// low float32 [T, H*dk + H*dv]: the decay's pre-activation, then the output gate's.
// conv float32 [C, taps] with C = 2*G*dk + H*dv (the filters of q, k, v stacked).
// state float32 [slots, state_stride]; the convolutions' inputs lie at conv_off as [taps - 1, C].
// prep float32 [T, prep_cols]: q | k | v | beta [H] | g [H*dk] | gate [H*dv].
// Units 0 .. 2G-1 are the heads of q and of k (convolution, silu, unit norm), units 2G .. 2G+H-1 the heads of v with that head's
// beta, decay and gate.
__device__ __forceinline__ float conv_at(const float* __restrict__ proj, const float* __restrict__ hist,
                                         const float* __restrict__ conv, int t, int i, int c, int C, int taps, int proj_cols) {
    float acc = 0.f;
    for (int j = 0; j < taps; ++j) {
        const int back = taps - 1 - j;
        const float x = (i - back >= 0) ? proj[static_cast<size_t>(t - back) * proj_cols + c]
                                        : hist[static_cast<size_t>(taps - 1 + i - back) * C + c];
        acc += conv[static_cast<size_t>(c) * taps + j] * x;
    }
    return acc;
}

// A workgroup a token and unit, a thread a channel: for steps of few tokens, which wait for memory once and not once a group of
// channels (twelve requests of 16 heads of 128 6.2 us, 9.3 by one wavefront a unit).
__global__ void delta_prepare_token_kernel(const float* __restrict__ proj, const float* __restrict__ low,
                                     const float* __restrict__ conv, const float* __restrict__ a_log,
                                     const float* __restrict__ dt_bias, float* __restrict__ state,
                                     const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ q_start,
                                     const int32_t* __restrict__ state_slot, float* __restrict__ prep,
                                     int G, int H, int dk, int dv, int taps, int proj_cols, size_t state_stride,
                                     size_t conv_off, int log_decay, int move_on) {
    __shared__ float scratch[16];
    const int t = blockIdx.x, unit = blockIdx.y;
    const int s = seq_of_token[t];
    const int i = t - q_start[s];              // place of the token in its portion
    const int QK = 2 * G * dk, C = QK + H * dv;
    const int prep_cols = C + H + H * dk + H * dv;
    float* hist = state + static_cast<size_t>(state_slot[s]) * state_stride + conv_off;
    float* out = prep + static_cast<size_t>(t) * prep_cols;
    // move_on: every sequence of the step brings one token, so the thread that has read a channel's last inputs is the
    // only one that does, and moves them on itself (no kernel of its own for that)
    auto moved = [&](int c) {
        for (int j = 0; j + 2 < taps; ++j) hist[static_cast<size_t>(j) * C + c] = hist[static_cast<size_t>(j + 1) * C + c];
        hist[static_cast<size_t>(taps - 2) * C + c] = proj[static_cast<size_t>(t) * proj_cols + c];
    };
    if (unit < 2 * G) {
        // a head of q or of k: every thread keeps its channels (dk <= 256 = threads)
        const int c = unit * dk + threadIdx.x;
        float y = 0.f;
        if (threadIdx.x < dk) {
            const float z = conv_at(proj, hist, conv, t, i, c, C, taps, proj_cols);
            y = silu_f(z);
            if (move_on && taps > 1) moved(c);
        }
        const float ss = block_sum(y * y, scratch);
        const float inv = (1.0f / sqrtf(ss + 1e-6f)) * (unit < G ? 1.0f / sqrtf(static_cast<float>(dk)) : 1.0f);
        if (threadIdx.x < dk) out[c] = y * inv;
        return;
    }
    const int h = unit - 2 * G;
    const float* prow = proj + static_cast<size_t>(t) * proj_cols;
    const float* lrow = low + static_cast<size_t>(t) * (H * dk + H * dv);
    for (int j = threadIdx.x; j < dv; j += blockDim.x) {
        const int c = QK + h * dv + j;
        const float z = conv_at(proj, hist, conv, t, i, c, C, taps, proj_cols);
        out[c] = silu_f(z);
        if (move_on && taps > 1) moved(c);
        out[C + H + H * dk + h * dv + j] = sigmoid_f(lrow[H * dk + h * dv + j]);
    }
    const float rate = expf(a_log[h]);
    for (int j = threadIdx.x; j < dk; j += blockDim.x) {
        const float z = lrow[h * dk + j] + dt_bias[h * dk + j];
        const float lg = -rate * softplus_f(z);
        out[C + H + h * dk + j] = log_decay ? lg : expf(lg);      // the chunked form sums logarithms
    }
    if (threadIdx.x == 0) out[C + h] = sigmoid_f(prow[C + h]);
}

// One wavefront a unit of four tokens: nothing meets in LDS, and four tokens of a sequence read the rows that their filters share
// once, all asked for together.  1,500 tokens of 16 heads of 128 (123 MB) took 65 us with a workgroup a token and unit, 43 now.
__global__ __launch_bounds__(256) void delta_prepare_kernel(const float* __restrict__ proj, const float* __restrict__ low,
                                     const float* __restrict__ conv, const float* __restrict__ a_log,
                                     const float* __restrict__ dt_bias, const float* __restrict__ state,
                                     const int32_t* __restrict__ seq_of_token, const int32_t* __restrict__ q_start,
                                     const int32_t* __restrict__ state_slot, float* __restrict__ prep,
                                     int T, int G, int H, int dk, int dv, int taps, int proj_cols, size_t state_stride,
                                     size_t conv_off, int log_decay) {
    constexpr int TOK = 4;
    const int lane = threadIdx.x & (WAVE - 1), unit = blockIdx.y;
    const int QK = 2 * G * dk, C = QK + H * dv;
    const int prep_cols = C + H + H * dk + H * dv;
    const int first = (blockIdx.x * 4 + threadIdx.x / WAVE) * TOK;
    // four tokens of one sequence behind its first three, filters of four: the seven rows that they need, all asked for at once
    if (first + 3 < T && taps == 4) {
        const int s = __builtin_amdgcn_readfirstlane(seq_of_token[first]);
        if (s == __builtin_amdgcn_readfirstlane(seq_of_token[first + 3]) && first - q_start[s] >= 3) {
            const float* rows = proj + static_cast<size_t>(first) * proj_cols;
            float* to = prep + static_cast<size_t>(first) * prep_cols;
            const bool value = unit >= 2 * G;
            const int h = unit - 2 * G, width = value ? dv : dk, c0 = value ? QK + h * dv : unit * dk;
            auto filtered = [&](int c, float (&y)[4]) {
                float x[7], w[4];
#pragma unroll
                for (int b = 0; b < 7; ++b) x[b] = rows[static_cast<ptrdiff_t>(b - 3) * proj_cols + c];
#pragma unroll
                for (int b = 0; b < 4; ++b) w[b] = conv[static_cast<size_t>(c) * 4 + b];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float acc = 0.f;
#pragma unroll
                    for (int b = 0; b < 4; ++b) acc += w[b] * x[j + b];
                    y[j] = silu_f(acc);
                }
            };
            if (!value) {
                float y[4][4], ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (b * WAVE >= dk) break;
                    const int at = lane + b * WAVE;
                    filtered(c0 + min(at, dk - 1), y[b]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) ss[j] += at < dk ? y[b][j] * y[b][j] : 0.f;
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    ss[j] = (1.0f / sqrtf(wave_sum(ss[j]) + 1e-6f)) * (unit < G ? 1.0f / sqrtf(static_cast<float>(dk)) : 1.0f);
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (lane + b * WAVE < dk) to[static_cast<size_t>(j) * prep_cols + c0 + lane + b * WAVE] = y[b][j] * ss[j];
                return;
            }
            const int wide = H * dk + H * dv;
            const float* lows = low + static_cast<size_t>(first) * wide;
            for (int at = lane; at < width; at += WAVE) {
                float y[4], gate[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) gate[j] = lows[static_cast<size_t>(j) * wide + H * dk + h * dv + at];
                filtered(c0 + at, y);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    to[static_cast<size_t>(j) * prep_cols + c0 + at] = y[j];
                    to[static_cast<size_t>(j) * prep_cols + C + H + H * dk + h * dv + at] = sigmoid_f(gate[j]);
                }
            }
            const float rate = expf(a_log[h]);
            for (int at = lane; at < dk; at += WAVE) {
                float z[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) z[j] = lows[static_cast<size_t>(j) * wide + h * dk + at];
                const float bias = dt_bias[h * dk + at];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float lg = -rate * softplus_f(z[j] + bias);
                    to[static_cast<size_t>(j) * prep_cols + C + H + h * dk + at] = log_decay ? lg : expf(lg);
                }
            }
            if (lane < 4) to[static_cast<size_t>(lane) * prep_cols + C + h] = sigmoid_f(rows[static_cast<size_t>(lane) * proj_cols + C + h]);
            return;
        }
    }
    for (int j = 0; j < TOK; ++j) {
        const int t = first + j;
        if (t >= T) return;
        const int s = seq_of_token[t];
        const int i = t - q_start[s];              // place of the token in its portion
        const float* hist = state + static_cast<size_t>(state_slot[s]) * state_stride + conv_off;
        float* out = prep + static_cast<size_t>(t) * prep_cols;
        if (unit < 2 * G) {
            // a head of q or of k: every lane keeps its channels (dk <= 256)
            float y[4], ss = 0.f;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int at = lane + b * WAVE;
                y[b] = 0.f;
                if (at < dk) {
                    const int c = unit * dk + at;
                    y[b] = silu_f(conv_at(proj, hist, conv, t, i, c, C, taps, proj_cols));
                }
                ss += y[b] * y[b];
            }
            ss = wave_sum(ss);
            const float inv = (1.0f / sqrtf(ss + 1e-6f)) * (unit < G ? 1.0f / sqrtf(static_cast<float>(dk)) : 1.0f);
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (lane + b * WAVE < dk) out[unit * dk + lane + b * WAVE] = y[b] * inv;
            continue;
        }
        const int h = unit - 2 * G;
        const float* prow = proj + static_cast<size_t>(t) * proj_cols;
        const float* lrow = low + static_cast<size_t>(t) * (H * dk + H * dv);
        for (int at = lane; at < dv; at += WAVE) {
            const int c = QK + h * dv + at;
            out[c] = silu_f(conv_at(proj, hist, conv, t, i, c, C, taps, proj_cols));
            out[C + H + H * dk + h * dv + at] = sigmoid_f(lrow[H * dk + h * dv + at]);
        }
        const float rate = expf(a_log[h]);
        for (int at = lane; at < dk; at += WAVE) {
            const float lg = -rate * softplus_f(lrow[h * dk + at] + dt_bias[h * dk + at]);
            out[C + H + h * dk + at] = log_decay ? lg : expf(lg);      // the chunked form sums logarithms
        }
        if (lane == 0) out[C + h] = sigmoid_f(prow[C + h]);
    }
}

__global__ void conv_state_update_kernel(const float* __restrict__ proj, float* __restrict__ state,
                                         const int32_t* __restrict__ q_start, const int32_t* __restrict__ q_len,
                                         const int32_t* __restrict__ state_slot, int C, int taps, int proj_cols,
                                         size_t state_stride, size_t conv_off) {
    const int s = blockIdx.x;
    const int n = q_len[s], first = q_start[s];
    float* hist = state + static_cast<size_t>(state_slot[s]) * state_stride + conv_off;
    for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < C; c += gridDim.y * blockDim.x) {
        // ascending j: entry j + n is read before any entry at or beyond it is written
        for (int j = 0; j < taps - 1; ++j) {
            const int i = n - (taps - 1) + j;
            hist[static_cast<size_t>(j) * C + c] = i >= 0 ? proj[static_cast<size_t>(first + i) * proj_cols + c]
                                                           : hist[static_cast<size_t>(j + n) * C + c];
        }
    }
}

// One workgroup: COLS = 256 / PARTS value channels of one head of one sequence.  The operands of CHUNK tokens at a
// time (q, k and g of the head, the workgroup's channels of v, beta) are brought into LDS by all threads together
// while the chunk before is worked through: the recurrence itself then waits for no load from memory, which at one
// token after the other would cost a round trip each.
__global__ void __launch_bounds__(256)
delta_rule_kernel(const float* __restrict__ prep, float* __restrict__ state, const int32_t* __restrict__ q_start,
                  const int32_t* __restrict__ q_len, const int32_t* __restrict__ state_slot, float* __restrict__ o,
                  int G, int H, int dv, size_t state_stride) {
    constexpr int DK = KPT * PARTS, COLS = 256 / PARTS;
    constexpr int CHUNK = DK <= 128 ? 16 : 8;
    constexpr int ROW = 3 * DK + COLS + 1;                    // q | k | g | v of the workgroup's channels | beta
    constexpr int LOADS = (CHUNK * ROW + 255) / 256;
    __shared__ float buf[2][CHUNK * ROW];
    const int s = blockIdx.x, h = blockIdx.y;
    const int part = threadIdx.x % PARTS;
    const int col0 = blockIdx.z * COLS;
    const int lcol = threadIdx.x / PARTS, col = col0 + lcol;
    const bool live = col < dv;
    const int g = h / (H / G);
    const int QK = 2 * G * DK, C = QK + H * dv;
    const int prep_cols = C + H + H * DK + H * dv;
    const int n = q_len[s], first = q_start[s];
    const float* rows = prep + static_cast<size_t>(first) * prep_cols;
    float* S_mem = state + static_cast<size_t>(state_slot[s]) * state_stride +
                   (static_cast<size_t>(h) * dv + (live ? col : 0)) * DK + part * KPT;
    float S[KPT];
#pragma unroll
    for (int i = 0; i < KPT; ++i) S[i] = live ? S_mem[i] : 0.f;

    float stage[LOADS];
    auto fetch = [&](int t0) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int e = threadIdx.x + j * 256;
            const int tok = e / ROW, r = e % ROW;
            float v = 0.f;
            if (e < CHUNK * ROW && t0 + tok < n) {
                const float* row = rows + static_cast<size_t>(t0 + tok) * prep_cols;
                if (r < DK) v = row[g * DK + r];
                else if (r < 2 * DK) v = row[G * DK + g * DK + (r - DK)];
                else if (r < 3 * DK) v = row[C + H + h * DK + (r - 2 * DK)];
                else if (r < 3 * DK + COLS) { if (col0 + (r - 3 * DK) < dv) v = row[QK + h * dv + col0 + (r - 3 * DK)]; }
                else v = row[C + h];
            }
            stage[j] = v;
        }
    };
    auto put = [&](float* dst) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const int e = threadIdx.x + j * 256;
            if (e < CHUNK * ROW) dst[e] = stage[j];
        }
    };
    fetch(0);
    put(buf[0]);
    __syncthreads();
    int which = 0;
    for (int t0 = 0; t0 < n; t0 += CHUNK) {
        const bool more = t0 + CHUNK < n;
        if (more) fetch(t0 + CHUNK);
        const float* cur = buf[which];
        const int count = min(CHUNK, n - t0);
        // unrolled, so that the reads from LDS and the products that do not wait for the memory (k . q) of the next
        // tokens stand ahead of the chain S -> S^T k -> u -> S that every token has to wait for
#pragma unroll 4
        for (int tt = 0; tt < count; ++tt) {
            const float* r = cur + tt * ROW;
            float a = 0.f, a1 = 0.f, b = 0.f, kq = 0.f, k[KPT];
#pragma unroll
            for (int i = 0; i < KPT; ++i) {
                const float q = r[part * KPT + i];
                k[i] = r[DK + part * KPT + i];
                S[i] *= r[2 * DK + part * KPT + i];
                if (i & 1) a1 += S[i] * k[i]; else a += S[i] * k[i];      // two chains of half the length
                b += S[i] * q;
                kq += k[i] * q;
            }
            a = parts_sum<PARTS>(a + a1);
            b = parts_sum<PARTS>(b);
            kq = parts_sum<PARTS>(kq);
            const float u = r[3 * DK + COLS] * (r[3 * DK + lcol] - a);
#pragma unroll
            for (int i = 0; i < KPT; ++i) S[i] += k[i] * u;
            if (live && part == 0) o[(static_cast<size_t>(first) + t0 + tt) * (H * dv) + h * dv + col] = b + u * kq;
        }
        if (more) put(buf[which ^ 1]);
        __syncthreads();
        which ^= 1;
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < KPT; ++i) S_mem[i] = S[i];
    }
}

// ------------------------------------------------------------------ sixteen tokens at a time
// Within a run of C = 16 tokens that starts from the memory S0, with L_t the sum of the logarithms of the decays
// of the run's tokens up to t (a vector over the key channels):
//     u_t + beta_t sum_{s<t} A_ts u_s = beta_t (v_t - S0^T (e^{L_t} k_t)),   A_ts = sum_c k_t[c] k_s[c] e^{L_t[c] - L_s[c]}
//     o_t = S0^T (e^{L_t} q_t) + sum_{s<=t} P_ts u_s,                        P_ts = sum_c q_t[c] k_s[c] e^{L_t[c] - L_s[c]}
//     S_C = diag(e^{L_C}) S0 + sum_s (e^{L_C - L_s} k_s) u_s^T
// Every exponent is a difference that is at most zero: nothing is divided by a decay, however small it gets.
// A, P, the inverse Tm = (I + diag(beta) tril(A, -1))^-1 diag(beta), its products with V and with Kt (the rows e^{L_t} k_t), and the
// scaled copies of k and q do not depend on the memory: delta_chunk_prepare makes them for all runs of the step at once.  What is
// left for the chain from run to run is
//     U = Tm V - (Tm Kt) S0;  O = Qt S0 + P U;  S <- diag(e^{L_C}) S0 + Kb^T U,
// which delta_chunk_scan does with v_mfma_f32_16x16x4_f32 (true 32-bit products and sums), one workgroup a
// (sequence, head, sixteen value channels) with its [DK, 16] piece of S in the accumulators' layout for the whole
// step.  A lane of that layout holds channels 4 (lane / 16) + r, r = 0..3, of each sixteen; as the second operand
// of a product over channels the four registers are used one after the other, and the first operand is read in
// the matching order (channel 4 (lane / 16) + r at step r), so that S never moves between layouts.
// Tokens past a sequence's end count as k = q = v = 0, beta = 0, decay 1: they leave S as it is.
// Runs are stored by slot = q_start / 16 + sequence + run: no two sequences of a step share one.
typedef float floatx4_t __attribute__((ext_vector_type(4)));
constexpr int RUN = 16;

// What is prepared for a run of tokens and a head, by place (floats): Tm Kt and Qt as [token][channel], Kb as [channel][token], P as
// [token][token], e^{L_C}, and Tm V as [value channel][token], the channels filled up to sixteens.
template <int DK> struct RunPlaces {
    static constexpr int tk = 0, qt = RUN * DK, kb = 2 * RUN * DK, p = 3 * RUN * DK, dec = p + RUN * RUN, tv = dec + DK;
};
__host__ __device__ constexpr int chunk_floats(int dk, int dv) { return 3 * RUN * dk + RUN * RUN + dk + RUN * ((dv + RUN - 1) / RUN * RUN); }

// The sequence of workgroup (x, u) of B x any: workgroups are dealt to the eight dies in turn, so with x itself a sequence's workgroups
// would lie on 8 / gcd(B, 8) of them, the ones of a long portion beside 7, 15, 23 or 31 single tokens all on one.  Every
// 8 / gcd(B, 8) values of u the sequences move on by one.  A float32 step of 481 tokens beside 31 single ones, six such layers: 7,920 -> 4,219 us,
// 300 beside 7 3,511 -> 3,207; beside 30 (no common factor) 3,833 : 3,844.
__device__ __forceinline__ int dealt_sequence(int x, int u, int B) {
    const int g = min(B & -B, 8), s = x - (u / (8 / g) & (g - 1));
    return s < 0 ? s + B : s;
}

__global__ void __launch_bounds__(256)
delta_chunk_prepare_kernel(const float* __restrict__ prep, float* __restrict__ chunks, const int32_t* __restrict__ q_start,
                           const int32_t* __restrict__ q_len, int G, int H, int dv) {
    constexpr int DK = KPT * PARTS, LD = DK + 4;
    using At = RunPlaces<DK>;
    __shared__ __attribute__((aligned(16))) float Ls[RUN * LD], ks[RUN * LD], qs[RUN * LD];
    __shared__ float As[RUN * (RUN + 1)], betas[RUN];
    __shared__ __attribute__((aligned(16))) float Tm[RUN * RUN];
    const int s = dealt_sequence(blockIdx.x, blockIdx.y + gridDim.y * blockIdx.z, gridDim.x), h = blockIdx.z;
    const int n = q_len[s], first = q_start[s];
    const int t0 = blockIdx.y * RUN;
    if (t0 >= n) return;
    const int g = h / (H / G);
    const int QK = 2 * G * DK, C = QK + H * dv;
    const int prep_cols = C + H + H * DK + H * dv;
    const size_t slot = static_cast<size_t>(first / RUN + s + blockIdx.y);
    float* out = chunks + (slot * H + h) * chunk_floats(DK, dv);
    const float* rows = prep + static_cast<size_t>(first + t0) * prep_cols;
    for (int e = threadIdx.x; e < RUN * DK; e += 256) {
        const int t = e / DK, c = e % DK;
        const bool valid = t0 + t < n;
        const float* row = rows + static_cast<size_t>(t) * prep_cols;
        Ls[t * LD + c] = valid ? row[C + H + h * DK + c] : 0.f;
        ks[t * LD + c] = valid ? row[G * DK + g * DK + c] : 0.f;
        qs[t * LD + c] = valid ? row[g * DK + c] : 0.f;
    }
    if (threadIdx.x < RUN) betas[threadIdx.x] = t0 + threadIdx.x < n ? rows[static_cast<size_t>(threadIdx.x) * prep_cols + C + h] : 0.f;
    __syncthreads();
    if (threadIdx.x < DK) {
        float run = 0.f;
        for (int t = 0; t < RUN; ++t) {
            run += Ls[t * LD + threadIdx.x];
            Ls[t * LD + threadIdx.x] = run;
        }
    }
    __syncthreads();
    // A and P: two neighbouring threads a pair j < t, half of the channels each; the last sixteen threads the diagonal of P
    {
        float a = 0.f, p = 0.f;
        int t, j;
        if (threadIdx.x < RUN * (RUN - 1)) {
            const int pair = threadIdx.x / 2;
            t = static_cast<int>((sqrtf(8.f * pair + 1.f) + 1.f) * 0.5f);       // pairs t (t - 1) / 2 .. are those of t
            t -= t * (t - 1) / 2 > pair;
            t += t * (t + 1) / 2 <= pair;
            j = pair - t * (t - 1) / 2;
            constexpr int HALF = DK / 2;
            const float *lt = Ls + t * LD, *lj = Ls + j * LD, *kt = ks + t * LD, *kj = ks + j * LD, *qt = qs + t * LD;
            for (int c = (threadIdx.x & 1) * HALF; c < ((threadIdx.x & 1) + 1) * HALF; c += 4) {
                const float4 l0 = *reinterpret_cast<const float4*>(lt + c), l1 = *reinterpret_cast<const float4*>(lj + c);
                const float4 k0 = *reinterpret_cast<const float4*>(kt + c), k1 = *reinterpret_cast<const float4*>(kj + c);
                const float4 q0 = *reinterpret_cast<const float4*>(qt + c);
                const float w[4] = {exp_below(l0.x - l1.x) * k1.x, exp_below(l0.y - l1.y) * k1.y, exp_below(l0.z - l1.z) * k1.z, exp_below(l0.w - l1.w) * k1.w};
                a += k0.x * w[0]; a += k0.y * w[1]; a += k0.z * w[2]; a += k0.w * w[3];
                p += q0.x * w[0]; p += q0.y * w[1]; p += q0.z * w[2]; p += q0.w * w[3];
            }
            a += __shfl_xor(a, 1, WAVE);
            p += __shfl_xor(p, 1, WAVE);
            if ((threadIdx.x & 1) == 0) {
                As[t * (RUN + 1) + j] = a;
                out[At::p + t * RUN + j] = p;
                out[At::p + j * RUN + t] = 0.f;
            }
        } else {
            t = threadIdx.x - RUN * (RUN - 1);
            for (int c = 0; c < DK; ++c) p += qs[t * LD + c] * ks[t * LD + c];
            out[At::p + t * RUN + t] = p;
        }
    }
    __syncthreads();
    // the scaled copies; what Kt needs stays where k was
    for (int e = threadIdx.x; e < RUN * DK; e += 256) {
        const int t = e / DK, c = e % DK;
        const float lt = Ls[t * LD + c], lc = Ls[(RUN - 1) * LD + c], k = ks[t * LD + c];
        const float grow = exp_below(lt);
        out[At::qt + e] = grow * qs[t * LD + c];
        ks[t * LD + c] = grow * k;
        qs[t * LD + c] = exp_below(lc - lt) * k;
        if (t == RUN - 1) out[At::dec + c] = grow;
    }
    if (threadIdx.x < RUN) {
        // column j of (I + diag(beta) tril(A, -1))^-1 diag(beta), from the top down
        const int j = threadIdx.x;
        float x[RUN];
#pragma unroll
        for (int t = 0; t < RUN; ++t) {
            float acc = 0.f;
#pragma unroll
            for (int r = 0; r < t; ++r) acc += As[t * (RUN + 1) + r] * x[r];
            x[t] = (t == j ? betas[j] : 0.f) - betas[t] * acc;
        }
#pragma unroll
        for (int t = 0; t < RUN; ++t) Tm[t * RUN + j] = x[t];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < RUN * DK; e += 256) out[At::kb + e] = qs[e % RUN * LD + e / RUN];
    // Tm Kt and Tm V: four tokens of a column a thread
    const int dvp = (dv + RUN - 1) / RUN * RUN;
    for (int e = threadIdx.x; e < 4 * (DK + dvp); e += 256) {
        const bool key = e < 4 * DK;
        const int part = key ? e / DK : (e - 4 * DK) / dvp, c = key ? e % DK : (e - 4 * DK) % dvp;
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int r = 0; r < RUN; ++r) {
            float x;
            if (key) x = ks[r * LD + c];
            else x = c < dv && t0 + r < n ? rows[static_cast<size_t>(r) * prep_cols + QK + h * dv + c] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) sum[i] += Tm[(4 * part + i) * RUN + r] * x;
        }
        if (key) {
#pragma unroll
            for (int i = 0; i < 4; ++i) out[At::tk + (4 * part + i) * DK + c] = sum[i];
        } else {
            *reinterpret_cast<float4*>(out + At::tv + c * RUN + 4 * part) = make_float4(sum[0], sum[1], sum[2], sum[3]);
        }
    }
}

// The key channels of a (head, sixteen value channels) are dealt to SCAN_WAVES wavefronts, sixteen at a time: each
// keeps its channels' rows of S and makes its share of (Tm Kt) S0 and Qt S0.  The shares of U meet in LDS once a run (two
// buffers in turn, so one barrier a run is enough: a wavefront can be one run ahead of another, never two); every
// wavefront then sums them in the same order, so all hold the same U, and moves its own rows of S on.  The shares of O, with
// a share of P U each, meet at the barrier of the run behind.
//
// What bounds it is the chain from run to run (128 workgroups for one prompt through 16 heads of 128 value channels): the
// products with S, the meeting in LDS and the update of S.  So nothing else stands in it: Tm is multiplied in beforehand, sums
// over channels go in two chains, the read-out fills the wait for the meeting, and the operands are asked for AHEAD runs
// before their turn (they come from beyond the L2 of most XCDs, which takes longer than a run).  1,500 tokens of 16 heads
// of 128 by 128 channels 145 -> 96 us (with operands at hand it takes 70, of which 25 matrix instructions a run are 31), while
// delta_chunk_prepare, which has Tm's products to make now and does half as many exponentials, takes 45 -> 48.
constexpr int scan_waves(int kt) { return kt % 4 == 0 ? 4 : kt % 2 == 0 ? 2 : 1; }

template <int KTW, int MINE> struct RunOperands {
    floatx4_t tk[KTW], qt[KTW], kb[KTW], dec[KTW];   // rows (lane % 16) of Tm Kt and Qt, channels 16 kt + 4 (lane / 16) + r; Kb of channel
                                                     // 16 kt + lane % 16, tokens 4 (lane / 16) + r; e^{L_C} of the lane's channels of S
    floatx4_t tv;                                    // Tm V of tokens 4 (lane / 16) + r, the lane's value channel
    float p[MINE];                                   // row (lane % 16) of P, columns 4 (lane / 16) + wave + waves * j
};

constexpr int SCAN_TILES = KPT * PARTS / RUN > 0 ? KPT * PARTS / RUN : 1, SCAN_WAVES = scan_waves(SCAN_TILES);

// (Three wavefronts a SIMD hold the operands of two runs up to two sixteens of channels each.  With two and three runs ahead one portion
// of 1,500 tokens takes as long, 94 us, and steps of many requests more: 300 tokens beside 40 single ones 73.6 us, now 67.6.)
__global__ void __launch_bounds__(64 * SCAN_WAVES) __attribute__((amdgpu_waves_per_eu(SCAN_TILES / SCAN_WAVES <= 2 ? 3 : 2)))
delta_chunk_scan_kernel(const float* __restrict__ chunks, float* __restrict__ state, const int32_t* __restrict__ q_start,
                        const int32_t* __restrict__ q_len, const int32_t* __restrict__ state_slot, float* __restrict__ o, int H, int dv,
                        size_t state_stride) {
    constexpr int DK = KPT * PARTS, SW = SCAN_WAVES, KTW = SCAN_TILES / SW, MINE = 4 / SW;
    constexpr int AHEAD = 2;
    using At = RunPlaces<DK>;
    __shared__ floatx4_t ushare[2][SW][WAVE], oshare[2][SW][WAVE];
    const int s = dealt_sequence(blockIdx.x, blockIdx.y + gridDim.y * blockIdx.z, gridDim.x), h = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int i = lane & 15, g4 = lane >> 4;
    const int col = blockIdx.z * RUN + i;
    const bool live = col < dv;
    const int n = q_len[s], first = q_start[s];
    if (n <= 0) return;
    const int ch0 = wave * KTW * RUN;                  // the wavefront's first key channel
    float* S_mem = state + static_cast<size_t>(state_slot[s]) * state_stride + (static_cast<size_t>(h) * dv + (live ? col : 0)) * DK + ch0 + 4 * g4;
    floatx4_t S[KTW];
#pragma unroll
    for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[kt][r] = live ? S_mem[kt * RUN + r] : 0.f;
    const char* base = reinterpret_cast<const char*>(chunks + (static_cast<size_t>(first / RUN + s) * H + h) * chunk_floats(DK, dv));
    const size_t per_run = static_cast<size_t>(H) * chunk_floats(DK, dv) * 4;
    // bytes from a run's beginning, the lane's part in 32 bits
    const uint32_t by_token = (i * DK + ch0 + 4 * g4) * 4, by_channel = ((ch0 + i) * RUN + 4 * g4) * 4, mine = (ch0 + 4 * g4) * 4;
    const uint32_t by_value = (col * RUN + 4 * g4) * 4, by_p = (i * RUN + 4 * g4) * 4;
    using Operands = RunOperands<KTW, MINE>;
    auto fetch = [&](Operands& x, int run) {
        const char* ch = base + per_run * run;
        auto load = [&](int place, uint32_t lane_part, int more) { return *reinterpret_cast<const floatx4_t*>(ch + place * 4 + lane_part + more); };
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt) {
            x.tk[kt] = load(At::tk, by_token, kt * RUN * 4);
            x.qt[kt] = load(At::qt, by_token, kt * RUN * 4);
            x.kb[kt] = load(At::kb, by_channel, kt * RUN * RUN * 4);
            x.dec[kt] = load(At::dec, mine, kt * RUN * 4);
        }
        x.tv = load(At::tv, by_value, 0);
#pragma unroll
        for (int j = 0; j < MINE; ++j) x.p[j] = *reinterpret_cast<const float*>(ch + (At::p + wave + SW * j) * 4 + by_p);
    };
    // the shares of a run's read-out, once all wavefronts have left them; a wavefront stores the tokens 4 (lane / 16) + r with r its own
    char* out = reinterpret_cast<char*>(o + static_cast<size_t>(first) * (H * dv) + h * dv);
    const uint32_t by_out = (4 * g4 * H * dv + col) * 4;
    auto read_out = [&](int run) {
#pragma unroll
        for (int j = 0; j < MINE; ++j) {
            const int r = wave + SW * j, tok = run * RUN + 4 * g4 + r;
            float val = 0.f;
#pragma unroll
            for (int w = 0; w < SW; ++w) val += reinterpret_cast<const float*>(&oshare[run & 1][w][lane])[r];
            if (live && tok < n) *reinterpret_cast<float*>(out + static_cast<size_t>(run * RUN + r) * (H * dv) * 4 + by_out) = val;
        }
    };
    const int runs = (n + RUN - 1) / RUN;
    Operands ops[AHEAD];
    auto step = [&](auto more, Operands& x, int run) {
        floatx4_t ua = {0.f, 0.f, 0.f, 0.f}, ub = {0.f, 0.f, 0.f, 0.f}, oa = ua, ob = ua;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int kt = 0; kt < KTW; ++kt) {
                floatx4_t& to = kt & 1 ? ub : ua;
                to = __builtin_amdgcn_mfma_f32_16x16x4f32(x.tk[kt][r], S[kt][r], to, 0, 0, 0);
            }
        ushare[run & 1][wave][lane] = ua + ub;
        __syncthreads();
        floatx4_t theirs[SW];
#pragma unroll
        for (int w = 0; w < SW; ++w) theirs[w] = ushare[run & 1][w][lane];
        __builtin_amdgcn_sched_barrier(0);
        // (the wait for them is filled with the read-out from S)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int kt = 0; kt < KTW; ++kt) {
                floatx4_t& to = kt & 1 ? ob : oa;
                to = __builtin_amdgcn_mfma_f32_16x16x4f32(x.qt[kt][r], S[kt][r], to, 0, 0, 0);
            }
        floatx4_t u = theirs[0];
#pragma unroll
        for (int w = 1; w < SW; ++w) u += theirs[w];
        u = x.tv - u;
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt) S[kt] *= x.dec[kt];
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int kt = 0; kt < KTW; ++kt) S[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.kb[kt][r], u[r], S[kt], 0, 0, 0);
        if (run > 0) read_out(run - 1);
#pragma unroll
        for (int j = 0; j < MINE; ++j) {
            float mine = u[SW * j];
#pragma unroll
            for (int w = 1; w < SW; ++w) mine = wave == w ? u[w + SW * j] : mine;
            oa = __builtin_amdgcn_mfma_f32_16x16x4f32(x.p[j], mine, oa, 0, 0, 0);
        }
        oshare[run & 1][wave][lane] = oa + ob;
        if constexpr (decltype(more)::value) fetch(x, min(run + AHEAD, runs - 1));
    };
    if (runs <= AHEAD) {
        // single tokens and short portions: their runs' operands once (asked for as in the loop, the last one's AHEAD times more, 8
        // single tokens beside 60 took 31 us, 200 beside 60 500; now 19 and 213)
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (j < runs) fetch(ops[j], j);
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (j < runs) step(std::false_type{}, ops[j], j);
    } else {
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) fetch(ops[j], j);
        int run = 0;
        for (; run + AHEAD <= runs; run += AHEAD) {
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) step(std::true_type{}, ops[j], run + j);
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (run + j < runs) step(std::false_type{}, ops[j], run + j);
    }
    __syncthreads();
    read_out(runs - 1);
    if (live) {
#pragma unroll
        for (int kt = 0; kt < KTW; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) S_mem[kt * RUN + r] = S[kt][r];
    }
}

// y[t, h, :] = o[t, h, :] / sqrt(mean(o[t, h, :]^2) + eps) * w * gate[t, h, :]; one wavefront a (token, head)
template <typename T>
__global__ void headnorm_gate_kernel(const float* __restrict__ o, const float* __restrict__ gate, size_t gate_stride,
                                     const float* __restrict__ w, T* __restrict__ y, int rows, int H, int dv, float eps) {
    const int lane = threadIdx.x & (WAVE - 1);
    const int r = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;      // t * H + h
    if (r >= rows) return;
    const int t = r / H, h = r % H;
    const float* orow = o + static_cast<size_t>(r) * dv;
    const float* grow = gate + static_cast<size_t>(t) * gate_stride + h * dv;
    float ss = 0.f;
    for (int c = lane; c < dv; c += WAVE) ss += orow[c] * orow[c];
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(dv) + eps);
    for (int c = lane; c < dv; c += WAVE) st(y + static_cast<size_t>(r) * dv + c, ((orow[c] * inv) * w[c]) * grow[c]);
}

NI_EXPORT int ni_delta_key_size() { return KPT * PARTS; }

NI_EXPORT int ni_delta_prepare(const void* proj, const void* low, const void* conv, const void* a_log, const void* dt_bias,
                               void* state, const void* seq_of_token, const void* q_start, const void* q_len,
                               const void* state_slot, void* prep, int T, int B, int G, int H, int dk, int dv, int taps,
                               int proj_cols, size_t state_stride, size_t conv_off, int log_decay, int max_q_len, hipStream_t stream) {
    if (T <= 0) return 0;
    const int move_on = max_q_len == 1;         // a step of single tokens: the prepare kernel moves the convolutions' inputs on
    if (dk != KPT * PARTS) return -1;
    const int C = 2 * G * dk + H * dv;
    if (dk > 256) return -2;
    // A wavefront takes four tokens where that still fills the chip and most groups of four lie in one sequence: 16 heads of 128, one
    // portion of 256 / 481 / 700 / 1,500 tokens (a token a workgroup : this) 15.3 : 17.6, 24.2 : 23.3, 32.6 : 27.3, 63.0 : 41.4; 300 beside 40
    // single tokens 18.6 : 24.9, 481 beside 31 25.8 : 41.9, 16 portions of 20 17.8 : 22.3.
    if (T >= 448 && T >= 64 * B && !move_on) {
        delta_prepare_kernel<<<dim3((T + 15) / 16, 2 * G + H), 256, 0, stream>>>((const float*)proj, (const float*)low, (const float*)conv,
                                                  (const float*)a_log, (const float*)dt_bias, (const float*)state,
                                                  (const int32_t*)seq_of_token, (const int32_t*)q_start,
                                                  (const int32_t*)state_slot, (float*)prep, T, G, H, dk, dv, taps, proj_cols,
                                                  state_stride, conv_off, log_decay);
    } else {
        const int widest = std::max(dk, std::min(dv, 256));
        delta_prepare_token_kernel<<<dim3(T, 2 * G + H), (widest + 63) / 64 * 64, 0, stream>>>((const float*)proj, (const float*)low, (const float*)conv,
                                                  (const float*)a_log, (const float*)dt_bias, (float*)state,
                                                  (const int32_t*)seq_of_token, (const int32_t*)q_start,
                                                  (const int32_t*)state_slot, (float*)prep, G, H, dk, dv, taps, proj_cols,
                                                  state_stride, conv_off, log_decay, move_on);
    }
    if (taps > 1 && !move_on) {
        dim3 grid(B, std::max(1, std::min(64, (C + 255) / 256)));
        conv_state_update_kernel<<<grid, 256, 0, stream>>>((const float*)proj, (float*)state, (const int32_t*)q_start,
                                                           (const int32_t*)q_len, (const int32_t*)state_slot, C, taps,
                                                           proj_cols, state_stride, conv_off);
    }
    return NI_LAUNCH_RESULT();
}

// floats of scratch that the chunked form needs per run of sixteen tokens and head (0: this key size has no such form);
// a step of T tokens in B sequences has at most T / 16 + B + 1 run slots
NI_EXPORT int ni_delta_run_floats(int dv) { return (KPT * PARTS) % RUN ? 0 : chunk_floats(KPT * PARTS, dv); }

// chunks: null for the token-by-token kernel (prep then holds the decays), else scratch for the chunked form
// (prep then holds the decays' logarithms); max_q_len is the longest portion of the step
NI_EXPORT int ni_delta_rule(const void* prep, void* chunks, void* state, const void* q_start, const void* q_len,
                            const void* state_slot, void* o, const void* norm_w, void* y, int T, int B, int max_q_len, int G,
                            int H, int dk, int dv, float eps, size_t state_stride, int dtype, hipStream_t stream) {
    if (T <= 0 || B <= 0) return 0;
    if (dk != KPT * PARTS) return -1;
    if (chunks) {
        if constexpr ((KPT * PARTS) % RUN == 0) {
            if (max_q_len < 1) return -1;
            const int runs = (max_q_len + RUN - 1) / RUN;
            delta_chunk_prepare_kernel<<<dim3(B, runs, H), 256, 0, stream>>>((const float*)prep, (float*)chunks, (const int32_t*)q_start,
                                                                             (const int32_t*)q_len, G, H, dv);
            delta_chunk_scan_kernel<<<dim3(B, H, (dv + RUN - 1) / RUN), 64 * SCAN_WAVES, 0, stream>>>(
                (const float*)chunks, (float*)state, (const int32_t*)q_start, (const int32_t*)q_len, (const int32_t*)state_slot,
                (float*)o, H, dv, state_stride);
        } else {
            return -3;
        }
    } else {
        constexpr int COLS = 256 / PARTS;
        dim3 grid(B, H, (dv + COLS - 1) / COLS);
        delta_rule_kernel<<<grid, 256, 0, stream>>>((const float*)prep, (float*)state, (const int32_t*)q_start,
                                                    (const int32_t*)q_len, (const int32_t*)state_slot, (float*)o, G, H, dv,
                                                    state_stride);
    }
    const int C = 2 * G * dk + H * dv;
    const int prep_cols = C + H + H * dk + H * dv;
    const float* gate = (const float*)prep + C + H + H * dk;
    const int rows = T * H;
    if (dtype == 0)
        headnorm_gate_kernel<float><<<(rows + 3) / 4, 256, 0, stream>>>((const float*)o, gate, prep_cols, (const float*)norm_w,
                                                                        (float*)y, rows, H, dv, eps);
    else
        headnorm_gate_kernel<bf16_t><<<(rows + 3) / 4, 256, 0, stream>>>((const float*)o, gate, prep_cols, (const float*)norm_w,
                                                                         (bf16_t*)y, rows, H, dv, eps);
    return NI_LAUNCH_RESULT();
}
