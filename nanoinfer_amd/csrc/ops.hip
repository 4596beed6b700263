// Row-wise and element-wise kernels of a decoder step for gfx950: embedding gather,
// residual-add + RMSNorm, rotation table, rotation + paged key/value write, SwiGLU.
//
// Conventions shared by all of them:
//   * the residual stream is float32; activations that feed a matrix product are the
//     compute type (float or bfloat16); all arithmetic is float32;
//   * a key/value pool is laid out [page, kv_head, slot_in_page, head_dim];
//   * every entry point is extern "C", takes raw device pointers and a hipStream_t, and
//     returns 0 or the hipError_t of its launch.  Shapes are checked by the host wrapper.
#include "common.h"
#include "pair_rows.h"

#include <algorithm>

// ---------------------------------------------------------------- embedding
// out[t, :] = table[ids[t], :]   (src/op/kernels/cuda/embedding_kernel.cu:30-48 of the reference;
// ids are range-checked on the host before upload, an id outside the table never reaches here.)
template <typename T>
__global__ void embedding_kernel(const int32_t* __restrict__ ids, const T* __restrict__ table,
                                 float* __restrict__ out, int d, int vocab) {
    const int t = blockIdx.x;
    int id = ids[t];
    if (id < 0 || id >= vocab) return;  // unreachable after the host check; never read out of bounds
    const T* row = table + static_cast<size_t>(id) * d;
    float* o = out + static_cast<size_t>(t) * d;
    for (int i = threadIdx.x; i < d; i += blockDim.x) o[i] = ld(row + i);
}

// ---------------------------------------------------------------- add + RMSNorm
// v = h[row] + pending[row];  out = v * rsqrt(mean(v^2) + eps) * w
// Without `rows` the sum is written back to h (the residual stream moves on) and out has T rows.
// With `rows` (a gather before the output head) h is left alone and out row r comes from h[rows[r]].
// Formula: src/op/kernels/cuda/rmsnorm_kernel.cu:50-103 of the reference.
// Rows of up to NV * blockDim elements are held in registers: every load of the row is issued
// before anything waits, and the row is read from memory once.
template <typename TP, typename TO, int NV>
__global__ void add_rmsnorm_kernel(float* __restrict__ h, const TP* __restrict__ pending, int addends, size_t addend_stride,
                                   const float* __restrict__ w, TO* __restrict__ out,
                                   const int32_t* __restrict__ rows, int d, float eps) {
    __shared__ float scratch[16];
    const int r = blockIdx.x;
    const size_t src = rows ? static_cast<size_t>(rows[r]) : static_cast<size_t>(r);
    float* hrow = h + src * d;
    const TP* prow = pending ? pending + src * d : nullptr;
    float v[NV], wv[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = threadIdx.x + j * blockDim.x;
        v[j] = i < d ? hrow[i] : 0.f;
        wv[j] = i < d ? w[i] : 0.f;
    }
    if (prow) {
        // several addends (the shares of a product whose K range was cut) are added in their order;
        // four at a time are asked for before any is added, so that their loads overlap
        for (int a0 = 0; a0 < addends; a0 += 4) {
            float t[4][NV];
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int j = 0; j < NV; ++j) {
                    const int i = threadIdx.x + j * blockDim.x;
                    t[b][j] = (a0 + b < addends && i < d) ? ld(prow + (a0 + b) * addend_stride + i) : 0.f;
                }
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int j = 0; j < NV; ++j) v[j] += t[b][j];
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) ss += v[j] * v[j];
    if (!rows && prow) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int i = threadIdx.x + j * blockDim.x;
            if (i < d) hrow[i] = v[j];
        }
    }
    ss = block_sum(ss, scratch);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
    TO* orow = out + static_cast<size_t>(r) * d;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = threadIdx.x + j * blockDim.x;
        if (i < d) st(orow + i, (v[j] * inv) * wv[j]);
    }
}

// The same for rows whose width is a multiple of four: a thread holds G groups of four consecutive
// elements, so that every access is 16 bytes of float32 or 8 bytes of bfloat16 a lane and neighbouring
// lanes touch neighbouring groups (a third of the instructions, and the memory system sees whole lines).
// HALVES (float32 rows of whole stages of 32 columns): the row is left as pairs of halves too (pair_rows.h), for the products behind
// the norm.  It is at hand here; a pass of its own reads it again and is a launch more: 512 rows of 2,048 behind two addends 8.2 + 5.4 us
// apart, 10.3 here; 1,500 rows 6.2 + 7.4 (that for each of two or three products) and 9.7.
template <typename TP, typename TO, int G, bool HALVES = false>
__global__ void add_rmsnorm_vec_kernel(float* __restrict__ h, const TP* __restrict__ pending, int addends, size_t addend_stride,
                                       const float* __restrict__ w, TO* __restrict__ out,
                                       const int32_t* __restrict__ rows, int d, float eps, char* __restrict__ planes = nullptr,
                                       int2* __restrict__ info = nullptr) {
    __shared__ float scratch[16];
    const int r = blockIdx.x;
    const size_t src = rows ? static_cast<size_t>(rows[r]) : static_cast<size_t>(r);
    float* hrow = h + src * d;
    const TP* prow = pending ? pending + src * d : nullptr;
    float v[G][4], wv[G][4];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int at = (threadIdx.x + g * blockDim.x) * 4;
        if (at < d) {
            VecIO<float, 4>::load(hrow + at, v[g]);
            VecIO<float, 4>::load(w + at, wv[g]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[g][e] = wv[g][e] = 0.f;
        }
    }
    if (prow) {
        // the addends in their order, four asked for before any is added
        for (int a0 = 0; a0 < addends; a0 += 4) {
            float t[4][G][4];
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const int at = (threadIdx.x + g * blockDim.x) * 4;
                    if (a0 + b < addends && at < d) {
                        VecIO<TP, 4>::load(prow + (a0 + b) * addend_stride + at, t[b][g]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) t[b][g][e] = 0.f;
                    }
                }
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int g = 0; g < G; ++g)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[g][e] += t[b][g][e];
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += v[g][e] * v[g][e];
    if (!rows && prow) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int at = (threadIdx.x + g * blockDim.x) * 4;
            if (at < d) store_packed<float, 4>(hrow + at, v[g]);
        }
    }
    ss = block_sum(ss, scratch);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
    TO* orow = out + static_cast<size_t>(r) * d;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int at = (threadIdx.x + g * blockDim.x) * 4;
        if (at < d) {
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[g][e] = y[e] = (v[g][e] * inv) * wv[g][e];
            store_packed<TO, 4>(orow + at, y);
        }
    }
    if constexpr (HALVES) {
        __shared__ uint32_t tops[16];
        __shared__ int bigs[16];
        const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, waves = blockDim.x / WAVE;
        uint32_t top = 0;
#pragma unroll
        for (int g = 0; g < G; ++g)
            if ((threadIdx.x + g * blockDim.x) * 4 < d)
#pragma unroll
                for (int e = 0; e < 4; ++e) top = max(top, __float_as_uint(v[g][e]) & 0x7fffffffu);
#pragma unroll
        for (int off = WAVE / 2; off > 0; off >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), off, WAVE)));
        if (lane == 0) tops[wave] = top;
        __syncthreads();
        for (int i = 0; i < waves; ++i) top = max(top, tops[i]);
        const int s = pair_scale(top);
        char* prow_out = planes + static_cast<size_t>(r) * d * 4;
        int big = 0;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int at = (threadIdx.x + g * blockDim.x) * 4;
            if (at < d) {
                float u[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    u[e] = ldexpf(v[g][e], s);
                    big += fabsf(u[e]) >= PAIR_BIG;
                }
                uint2 hh, ll;
                pair_up(u, hh, ll);
                *reinterpret_cast<uint2*>(prow_out + pair_place(at)) = hh;
                *reinterpret_cast<uint2*>(prow_out + pair_place(at) + 32) = ll;
            }
        }
#pragma unroll
        for (int off = WAVE / 2; off > 0; off >>= 1) big += __shfl_xor(big, off, WAVE);
        if (lane == 0) bigs[wave] = big;
        __syncthreads();
        if (threadIdx.x == 0) {
            big = 0;
            for (int i = 0; i < waves; ++i) big += bigs[i];
            info[r] = pair_row_info(s, top, big);
        }
    }
}

// Rows of any width: two passes over memory.
template <typename TP, typename TO>
__global__ void add_rmsnorm_wide_kernel(float* __restrict__ h, const TP* __restrict__ pending, int addends, size_t addend_stride,
                                        const float* __restrict__ w, TO* __restrict__ out,
                                        const int32_t* __restrict__ rows, int d, float eps) {
    __shared__ float scratch[16];
    const int r = blockIdx.x;
    const size_t src = rows ? static_cast<size_t>(rows[r]) : static_cast<size_t>(r);
    float* hrow = h + src * d;
    const TP* prow = pending ? pending + src * d : nullptr;
    float ss = 0.f;
    auto sum_at = [&](int i) {
        float v = hrow[i];
        if (prow)
            for (int a = 0; a < addends; ++a) v += ld(prow + a * addend_stride + i);
        return v;
    };
    for (int i = threadIdx.x; i < d; i += blockDim.x) {
        const float v = sum_at(i);
        if (!rows && prow) hrow[i] = v;
        ss += v * v;
    }
    ss = block_sum(ss, scratch);
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(d) + eps);
    TO* orow = out + static_cast<size_t>(r) * d;
    for (int i = threadIdx.x; i < d; i += blockDim.x) {
        const float v = (rows && prow) ? sum_at(i) : hrow[i];
        st(orow + i, (v * inv) * w[i]);
    }
}

// ---------------------------------------------------------------- rotation table
// cos/sin[pos, p] of the float32 product pos * inv_freq[p]
// (src/op/kernels/cuda/rope_kernel.cu:129-131 of the reference; the frequencies come from the host).
__global__ void rope_table_kernel(const float* __restrict__ inv_freq, float* __restrict__ cos_t,
                                  float* __restrict__ sin_t, int max_pos, int half) {
    size_t idx = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= static_cast<size_t>(max_pos) * half) return;
    int pos = static_cast<int>(idx / half);
    int p = static_cast<int>(idx % half);
    float angle = static_cast<float>(pos) * inv_freq[p];
    cos_t[idx] = cosf(angle);
    sin_t[idx] = sinf(angle);
}

// ---------------------------------------------------------------- rotation + key/value write
// qkv is [T, (H + 2*KVH) * hd]: q heads, then k heads, then v heads.  Queries are rotated in
// place; rotated keys and plain values go to the pools at slot_mapping[t] (= page*page_size + slot;
// negative: this layer does not write).  Pairs are (j, j + rot/2) inside the first `rot` dims of a
// head, which is the pairing of the checkpoint's row order (the reference permutes rows at export,
// tools/export_llama3.py:571-583, and rotates neighbours, src/op/kernels/cuda/rope_kernel.cu:32-84).
template <typename T>
__global__ void rope_kv_write_kernel(T* __restrict__ qkv, const int32_t* __restrict__ positions,
                                     const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                     const int32_t* __restrict__ slot_mapping, T* __restrict__ kpool,
                                     T* __restrict__ vpool, int H, int KVH, int hd, int rot, int page_size) {
    const int t = blockIdx.x;
    const int half = rot / 2;
    const int row_width = (H + 2 * KVH) * hd;
    T* row = qkv + static_cast<size_t>(t) * row_width;
    const int pos = positions[t];
    const float* c = cos_t ? cos_t + static_cast<size_t>(pos) * half : nullptr;
    const float* s = sin_t ? sin_t + static_cast<size_t>(pos) * half : nullptr;
    const int slot = slot_mapping ? slot_mapping[t] : -1;
    const int page = slot >= 0 ? slot / page_size : 0;
    const int off = slot >= 0 ? slot % page_size : 0;

    // q and k heads: rotate pairs; dims beyond `rot` pass through.
    const int per_head = hd - half;  // `half` pairs + (hd - rot) pass-through dims
    for (int item = threadIdx.x; item < (H + KVH) * per_head; item += blockDim.x) {
        const int head = item / per_head;
        const int j = item % per_head;
        T* hp = row + static_cast<size_t>(head) * hd;
        const bool is_k = head >= H;
        T* dst = nullptr;
        if (is_k && slot >= 0)
            dst = kpool + ((static_cast<size_t>(page) * KVH + (head - H)) * page_size + off) * hd;
        if (j < half) {
            float x0 = ld(hp + j), x1 = ld(hp + j + half);
            float cs = c[j], sn = s[j];
            float y0 = x0 * cs - x1 * sn;
            float y1 = x0 * sn + x1 * cs;
            if (!is_k) {
                st(hp + j, y0);
                st(hp + j + half, y1);
            } else if (dst) {
                st(dst + j, y0);
                st(dst + j + half, y1);
            }
        } else {
            const int dim = rot + (j - half);
            if (is_k && dst) dst[dim] = hp[dim];
        }
    }
    if (slot >= 0) {
        for (int item = threadIdx.x; item < KVH * hd; item += blockDim.x) {
            const int g = item / hd, dim = item % hd;
            vpool[((static_cast<size_t>(page) * KVH + g) * page_size + off) * hd + dim] =
                row[static_cast<size_t>(H + KVH + g) * hd + dim];
        }
    }
}

// ---------------------------------------------------------------- gated hidden units
// out[t, i] = act(gu[t, i]) * gu[t, I + i], act silu or gelu in its tanh form   (SwiGLU: src/op/kernels/cuda/swiglu_kernel.cu:31-39 of the
// reference, with expf instead of the fast intrinsic).
template <typename T>
__global__ void swiglu_kernel(const T* __restrict__ gu, T* __restrict__ out, int I, size_t n, GatedUnit unit) {
    size_t idx = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    size_t t = idx / I;
    int i = static_cast<int>(idx % I);
    float g = ld(gu + t * 2 * I + i);
    float u = ld(gu + t * 2 * I + I + i);
    st(out + idx, unit.value(g, u));
}

// The same in accesses of 16 bytes, for head sizes and rotated halves that are multiples of 16 bytes
// of elements: an item is one such piece of a pair of halves, of a key's unrotated dims, or of a value.
template <typename T>
__global__ void rope_kv_write_vec_kernel(T* __restrict__ qkv, const int32_t* __restrict__ positions,
                                         const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                         const int32_t* __restrict__ slot_mapping, T* __restrict__ kpool,
                                         T* __restrict__ vpool, int H, int KVH, int hd, int rot, int page_size) {
    constexpr int V = 16 / sizeof(T);
    typedef uint32_t u32x4_hw __attribute__((ext_vector_type(4)));
    const int t = blockIdx.x;
    const int half = rot / 2;
    T* row = qkv + static_cast<size_t>(t) * (H + 2 * KVH) * hd;
    const int pos = positions[t];
    const float* c = cos_t + static_cast<size_t>(pos) * half;
    const float* s = sin_t + static_cast<size_t>(pos) * half;
    const int slot = slot_mapping ? slot_mapping[t] : -1;
    const int page = slot >= 0 ? slot / page_size : 0;
    const int off = slot >= 0 ? slot % page_size : 0;
    const int rot_vecs = half / V, pass_vecs = (hd - rot) / V, head_vecs = hd / V;
    const int n_rot = (H + KVH) * rot_vecs;
    const int n_pass = slot >= 0 ? KVH * pass_vecs : 0;
    const int n_val = slot >= 0 ? KVH * head_vecs : 0;
    for (int item = threadIdx.x; item < n_rot + n_pass + n_val; item += blockDim.x) {
        if (item < n_rot) {
            const int head = item / rot_vecs, j = (item % rot_vecs) * V;
            T* hp = row + static_cast<size_t>(head) * hd;
            const bool is_k = head >= H;
            if (is_k && slot < 0) continue;
            T* dst = is_k ? kpool + ((static_cast<size_t>(page) * KVH + (head - H)) * page_size + off) * hd : hp;
            float x0[V], x1[V], cs[V], sn[V], y0[V], y1[V];
            VecIO<T, V>::load(hp + j, x0);
            VecIO<T, V>::load(hp + j + half, x1);
            VecIO<float, V>::load(c + j, cs);
            VecIO<float, V>::load(s + j, sn);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                y0[e] = x0[e] * cs[e] - x1[e] * sn[e];
                y1[e] = x0[e] * sn[e] + x1[e] * cs[e];
            }
            if constexpr (sizeof(T) == 4) {
                store_packed<T, 4>(dst + j, y0);
                store_packed<T, 4>(dst + j + half, y1);
            } else {
                store_packed<T, 8>(dst + j, y0);
                store_packed<T, 8>(dst + j + half, y1);
            }
        } else if (item < n_rot + n_pass) {
            const int k = item - n_rot, g = k / pass_vecs, dim = rot + (k % pass_vecs) * V;
            T* dst = kpool + ((static_cast<size_t>(page) * KVH + g) * page_size + off) * hd;
            *reinterpret_cast<u32x4_hw*>(dst + dim) = *reinterpret_cast<const u32x4_hw*>(row + static_cast<size_t>(H + g) * hd + dim);
        } else {
            const int k = item - n_rot - n_pass, g = k / head_vecs, dim = (k % head_vecs) * V;
            T* dst = vpool + ((static_cast<size_t>(page) * KVH + g) * page_size + off) * hd;
            *reinterpret_cast<u32x4_hw*>(dst + dim) =
                *reinterpret_cast<const u32x4_hw*>(row + static_cast<size_t>(H + KVH + g) * hd + dim);
        }
    }
}

// The same for a product that was cut along K: its shares' float32 sums [S][T][(H + 2 KVH) * hd] are added in their order, rotated and
// stored, the queries in rows of their own.  One pass instead of two (512 rows of the 1B shape in float32, four shares of 6 MB: 6.3 us for a
// kernel that adds them and 5.5 for the one above, 7.4 here): bound by the shares, which the caches hold.  Dims in vectors of four.
// SHARES: how many, known to the compiler, so that all are asked for at once; 0: `S`, by fours.  Six shares of 65 rows of [5120, 3072] in bfloat16, the
// product counted: 16.3 us, 21.8 where each waited for the one before; a kernel that adds them and the one above 18.6.
template <typename T, int SHARES>
__global__ __launch_bounds__(256) void rope_kv_write_shares_kernel(const float* __restrict__ parts, int S, T* __restrict__ q, const int32_t* __restrict__ positions,
                                                                   const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                                                   const int32_t* __restrict__ slot_mapping, T* __restrict__ kpool,
                                                                   T* __restrict__ vpool, int H, int KVH, int hd, int rot, int page_size) {
    constexpr int V = 4;
    const int t = blockIdx.x, half = rot / 2;
    const size_t width = static_cast<size_t>(H + 2 * KVH) * hd, share = gridDim.x * width;
    const float* row = parts + t * width;
    const int pos = positions[t];
    const int slot = slot_mapping ? slot_mapping[t] : -1;
    const int page = slot >= 0 ? slot / page_size : 0, off = slot >= 0 ? slot % page_size : 0;
    const int stored = H + (slot >= 0 ? 2 * KVH : 0);                  // heads that go somewhere
    const int rot_vecs = half / V, pass_vecs = (hd - rot) / V, head_vecs = hd / V;
    const int turned = min(stored, H + KVH), n_rot = turned * rot_vecs, n_pass = turned * pass_vecs;
    auto sum = [&](int at, float* v) {
        VecIO<float, V>::load(row + at, v);
        if constexpr (SHARES > 0) {
            float u[SHARES][V];
#pragma unroll
            for (int p = 1; p < SHARES; ++p) VecIO<float, V>::load(row + p * share + at, u[p]);
#pragma unroll
            for (int p = 1; p < SHARES; ++p)
#pragma unroll
                for (int e = 0; e < V; ++e) v[e] += u[p][e];
        } else {
            constexpr int EACH = 4;
            int p = 1;
            for (; p + EACH <= S; p += EACH) {
                float u[EACH][V];
#pragma unroll
                for (int i = 0; i < EACH; ++i) VecIO<float, V>::load(row + (p + i) * share + at, u[i]);
#pragma unroll
                for (int i = 0; i < EACH; ++i)
#pragma unroll
                    for (int e = 0; e < V; ++e) v[e] += u[i][e];
            }
            for (; p < S; ++p) {
                float u[V];
                VecIO<float, V>::load(row + p * share + at, u);
#pragma unroll
                for (int e = 0; e < V; ++e) v[e] += u[e];
            }
        }
    };
    auto place = [&](int head) {
        if (head < H) return q + (static_cast<size_t>(t) * H + head) * hd;
        const int g = head < H + KVH ? head - H : head - H - KVH;
        return (head < H + KVH ? kpool : vpool) + ((static_cast<size_t>(page) * KVH + g) * page_size + off) * hd;
    };
    for (int item = threadIdx.x; item < n_rot + n_pass + (stored - turned) * head_vecs; item += 256) {
        if (item < n_rot) {
            const int head = item / rot_vecs, j = (item % rot_vecs) * V;
            float x0[V], x1[V], cs[V], sn[V], y0[V], y1[V];
            sum(head * hd + j, x0);
            sum(head * hd + j + half, x1);
            VecIO<float, V>::load(cos_t + static_cast<size_t>(pos) * half + j, cs);
            VecIO<float, V>::load(sin_t + static_cast<size_t>(pos) * half + j, sn);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                y0[e] = x0[e] * cs[e] - x1[e] * sn[e];
                y1[e] = x0[e] * sn[e] + x1[e] * cs[e];
            }
            T* dst = place(head);
            store_packed<T, V>(dst + j, y0);
            store_packed<T, V>(dst + j + half, y1);
        } else {
            const bool pass = item < n_rot + n_pass;
            const int k = item - n_rot - (pass ? 0 : n_pass), vecs = pass ? pass_vecs : head_vecs;
            const int head = k / vecs + (pass ? 0 : H + KVH), dim = (k % vecs) * V + (pass ? rot : 0);
            float v[V];
            sum(head * hd + dim, v);
            store_packed<T, V>(place(head) + dim, v);
        }
    }
}

// The same, 16 bytes of gate and of up per thread (rows whose width is a multiple of V elements).
// The bfloat16 instantiation takes the exponential with the hardware's exp2: its error is far
// below the rounding of the stored result.
template <typename T, int V>
__global__ void swiglu_vec_kernel(const T* __restrict__ gu, T* __restrict__ out, int I, size_t n_vec, GatedUnit unit) {
    const size_t idx = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (idx >= n_vec) return;
    const int per_row = I / V;
    const size_t t = idx / per_row;
    const int i = static_cast<int>(idx % per_row) * V;
    float g[V], u[V], y[V];
    VecIO<T, V>::load(gu + t * 2 * I + i, g);
    VecIO<T, V>::load(gu + t * 2 * I + I + i, u);
#pragma unroll
    for (int e = 0; e < V; ++e) y[e] = sizeof(T) == 2 ? unit.rough(g[e], u[e]) : unit.value(g[e], u[e]);
    VecIO<T, V>::store(out + t * I + i, y);
}

// ---------------------------------------------------------------- random weights
// Element `start + i` of the normal stream of `key`: a counter-based generator (splitmix64 over
// key + (index + 1) * gamma, Box-Muller over two 24-bit fractions).  Every operation is an IEEE
// float32 operation rounded on its own (contraction into fused multiply-adds is switched off in
// these routines; division and square root are the correctly rounded ones), and logarithm and
// cosine are fixed polynomials, so that the host's numpy twin of this routine
// (nanoinfer_amd/weights/random_init.py) gives the same bits.
__device__ __forceinline__ float rn_poly6(float x2, float c0, float c1, float c2, float c3, float c4, float c5) {
#pragma clang fp contract(off)
    float acc = c5;
    acc = acc * x2; acc = acc + c4;
    acc = acc * x2; acc = acc + c3;
    acc = acc * x2; acc = acc + c2;
    acc = acc * x2; acc = acc + c1;
    acc = acc * x2; acc = acc + c0;
    return acc;
}

__device__ __forceinline__ float counter_normal(uint64_t key, uint64_t index, float mean, float std) {
#pragma clang fp contract(off)
    uint64_t z = key + (index + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    const int k1 = static_cast<int>(z >> 40) + 1;          // 1 .. 2^24
    const int k2 = static_cast<int>(z & 0xFFFFFFull);      // 0 .. 2^24 - 1
    // -2 ln(k1 / 2^24): k1 = m * 2^e, m brought into [sqrt(1/2), sqrt(2)); ln m = 2 atanh((m-1)/(m+1))
    int e;
    float m = frexpf(static_cast<float>(k1), &e);          // m in [0.5, 1), exact
    if (m < 0.7071067811865476f) { m = m * 2.0f; e -= 1; }
    const float ef = static_cast<float>(e - 24);
    const float num = m - 1.0f, den = m + 1.0f;
    const float s = num / den;                             // correctly rounded (the compiler's default for HIP)
    const float s2 = s * s;
    const float ln_m = s * rn_poly6(s2, 2.0f / 1, 2.0f / 3, 2.0f / 5, 2.0f / 7, 2.0f / 9, 2.0f / 11);
    const float e_ln2 = ef * 0.6931471805599453f;
    const float ln_u = e_ln2 + ln_m;
    const float radius = sqrtf(-2.0f * ln_u);              // correctly rounded as well
    // cos(2 pi k2 / 2^24): quarter turns q, the rest f in [0, 1) folded to [0, 1/2], x = pi/2 f
    const int q = k2 >> 22;
    const float f = static_cast<float>(k2 & 0x3FFFFF) * (1.0f / 4194304.0f);
    const bool fold = f > 0.5f;
    const float x = (fold ? 1.0f - f : f) * 1.5707963267948966f;
    const float x2 = x * x;
    const float sin_x = x * rn_poly6(x2, 1.0f, -1.0f / 6, 1.0f / 120, -1.0f / 5040, 1.0f / 362880, -1.0f / 39916800);
    const float cos_x = rn_poly6(x2, 1.0f, -0.5f, 1.0f / 24, -1.0f / 720, 1.0f / 40320, -1.0f / 3628800);
    const float sin_f = fold ? cos_x : sin_x;
    const float cos_f = fold ? sin_x : cos_x;
    const float c = q == 0 ? cos_f : q == 1 ? -sin_f : q == 2 ? -cos_f : sin_f;
    const float n = radius * c;
    const float scaled = std * n;
    return scaled + mean;
}

template <typename T>
__global__ void random_normal_kernel(T* __restrict__ out, size_t count, uint64_t key, uint64_t start, float mean, float std) {
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += stride)
        st(out + i, counter_normal(key, start + i, mean, std));
}

// ================================================================ entry points
// dtype codes: 0 = float32, 1 = bfloat16

static inline bool aligned_to(size_t bytes, const void* a, const void* b = nullptr, const void* c = nullptr,
                              const void* d = nullptr) {
    return (reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c) |
            reinterpret_cast<uintptr_t>(d)) % bytes == 0;
}

static inline unsigned blocks_for(size_t n, unsigned per) { return static_cast<unsigned>((n + per - 1) / per); }

NI_EXPORT int ni_embedding(const void* ids, const void* table, void* out, int T, int d, int vocab,
                           int table_dtype, hipStream_t stream) {
    if (T <= 0) return 0;
    if (table_dtype == 0)
        embedding_kernel<float><<<T, 256, 0, stream>>>((const int32_t*)ids, (const float*)table, (float*)out, d, vocab);
    else
        embedding_kernel<bf16_t><<<T, 256, 0, stream>>>((const int32_t*)ids, (const bf16_t*)table, (float*)out, d, vocab);
    return NI_LAUNCH_RESULT();
}

// Whether the norm of rows of d numbers takes a vector of four a thread instead of two: more wavefronts a row to wait with, half the
// chain in each.  Two : one (us, rows of 2,048 in bfloat16): 17 rows 3.7 : 3.2, 64 with four addends 3.8 : 3.3, 512 6.9 : 6.3, 2,045 19.2 : 18.2,
// of 3,072 at 17 / 512 / 2,045 rows 3.6 : 3.4, 5.6 : 5.5, 16.4 : 15.7; past 4,096 a workgroup has no more threads.  Float32 rows may be left as pairs
// of halves too, which keeps a thread at work: of 2,048 at 164 / 512 / 1,024 rows 5.4 : 4.7, 9.1 : 8.7, 13.2 : 13.0, but 1,500 12.1 : 13.0, and of 3,072
// at 512 8.1 : 8.7 (the norm that leaves none goes by the same line: the same bits).
static bool one_vector_a_thread(int d, int n_rows, bool float32) { return float32 ? d <= 2048 && n_rows <= 1024 : d <= 4096; }

template <typename TP, typename TO>
static void launch_add_rmsnorm(float* h, const TP* pending, int addends, size_t addend_stride, const float* w, TO* out,
                               const int32_t* rows, int n_rows, int d, float eps, hipStream_t stream) {
    constexpr int NV = 8;
    if (d <= NV * 1024) {
        const int threads = d <= NV * 64 ? 64 : d <= NV * 128 ? 128 : d <= NV * 256 ? 256 : d <= NV * 512 ? 512 : 1024;
        if (d % 4 == 0 && aligned_to(16, h, w) && aligned_to(4 * sizeof(TP), pending) && aligned_to(4 * sizeof(TO), out) &&
            (addends <= 1 || addend_stride % 4 == 0)) {
            if (one_vector_a_thread(d, n_rows, sizeof(TO) == 4)) {
                add_rmsnorm_vec_kernel<TP, TO, 1><<<n_rows, (d / 4 + WAVE - 1) / WAVE * WAVE, 0, stream>>>(h, pending, addends, addend_stride, w, out, rows, d, eps);
                return;
            }
            add_rmsnorm_vec_kernel<TP, TO, NV / 4><<<n_rows, threads, 0, stream>>>(h, pending, addends, addend_stride, w, out,
                                                                                  rows, d, eps);
            return;
        }
        add_rmsnorm_kernel<TP, TO, NV><<<n_rows, threads, 0, stream>>>(h, pending, addends, addend_stride, w, out, rows, d, eps);
    } else {
        add_rmsnorm_wide_kernel<TP, TO><<<n_rows, 1024, 0, stream>>>(h, pending, addends, addend_stride, w, out, rows, d, eps);
    }
}

// pending: null, or [T, d] of the output type, or (addends >= 1 with float_addends) float32 [addends, T, d], whose
// slices are added in their order.
NI_EXPORT int ni_add_rmsnorm(void* h, const void* pending, int addends, int float_addends, size_t addend_stride,
                             const void* w, void* out, const void* rows, int n_rows, int d, float eps, int dtype,
                             hipStream_t stream) {
    if (n_rows <= 0) return 0;
    if (pending && (addends < 1 || (addends > 1 && !float_addends))) return -1;
    if (dtype == 0)
        launch_add_rmsnorm<float, float>((float*)h, (const float*)pending, addends, addend_stride, (const float*)w,
                                         (float*)out, (const int32_t*)rows, n_rows, d, eps, stream);
    else if (float_addends)
        launch_add_rmsnorm<float, bf16_t>((float*)h, (const float*)pending, addends, addend_stride, (const float*)w,
                                          (bf16_t*)out, (const int32_t*)rows, n_rows, d, eps, stream);
    else
        launch_add_rmsnorm<bf16_t, bf16_t>((float*)h, (const bf16_t*)pending, addends, addend_stride, (const float*)w,
                                           (bf16_t*)out, (const int32_t*)rows, n_rows, d, eps, stream);
    return NI_LAUNCH_RESULT();
}

// The same for float32 rows, all of them, that are left as pairs of halves as well: d in whole stages of 32 columns, everything
// aligned to 16 bytes.
NI_EXPORT int ni_add_rmsnorm_halves(void* h, const void* pending, int addends, size_t addend_stride, const void* w, void* out, void* planes,
                                    void* info, int n_rows, int d, float eps, hipStream_t stream) {
    constexpr int NV = 8;
    if (n_rows <= 0) return 0;
    if (d <= 0 || d % 32 || d > NV * 1024 || (pending && addends < 1) || !aligned_to(16, h, w) || !aligned_to(16, pending, out) ||
        !aligned_to(16, planes) || (addends > 1 && addend_stride % 4))
        return static_cast<int>(hipErrorInvalidValue);
    const int threads = d <= NV * 64 ? 64 : d <= NV * 128 ? 128 : d <= NV * 256 ? 256 : d <= NV * 512 ? 512 : 1024;
    if (one_vector_a_thread(d, n_rows, true))
        add_rmsnorm_vec_kernel<float, float, 1, true><<<n_rows, (d / 4 + WAVE - 1) / WAVE * WAVE, 0, stream>>>(
            (float*)h, (const float*)pending, addends, addend_stride, (const float*)w, (float*)out, nullptr, d, eps, (char*)planes, (int2*)info);
    else add_rmsnorm_vec_kernel<float, float, NV / 4, true><<<n_rows, threads, 0, stream>>>(
        (float*)h, (const float*)pending, addends, addend_stride, (const float*)w, (float*)out, nullptr, d, eps, (char*)planes, (int2*)info);
    return NI_LAUNCH_RESULT();
}

NI_EXPORT int ni_rope_table(const void* inv_freq, void* cos_t, void* sin_t, int max_pos, int half,
                            hipStream_t stream) {
    size_t n = static_cast<size_t>(max_pos) * half;
    if (n == 0) return 0;
    rope_table_kernel<<<blocks_for(n, 256), 256, 0, stream>>>((const float*)inv_freq, (float*)cos_t, (float*)sin_t,
                                                              max_pos, half);
    return NI_LAUNCH_RESULT();
}

NI_EXPORT int ni_rope_kv_write(void* qkv, const void* positions, const void* cos_t, const void* sin_t,
                               const void* slot_mapping, void* kpool, void* vpool, int T, int H, int KVH, int hd,
                               int rot, int page_size, int dtype, hipStream_t stream) {
    if (T <= 0) return 0;
    const int vec = dtype == 0 ? 4 : 8;           // elements of a 16-byte access
    if (rot > 0 && hd % vec == 0 && (rot / 2) % vec == 0 && aligned_to(16, qkv, cos_t, sin_t) && aligned_to(16, kpool, vpool)) {
        if (dtype == 0)
            rope_kv_write_vec_kernel<float><<<T, 256, 0, stream>>>((float*)qkv, (const int32_t*)positions, (const float*)cos_t,
                                                                   (const float*)sin_t, (const int32_t*)slot_mapping,
                                                                   (float*)kpool, (float*)vpool, H, KVH, hd, rot, page_size);
        else
            rope_kv_write_vec_kernel<bf16_t><<<T, 256, 0, stream>>>((bf16_t*)qkv, (const int32_t*)positions,
                                                                    (const float*)cos_t, (const float*)sin_t,
                                                                    (const int32_t*)slot_mapping, (bf16_t*)kpool,
                                                                    (bf16_t*)vpool, H, KVH, hd, rot, page_size);
        return NI_LAUNCH_RESULT();
    }
    if (dtype == 0)
        rope_kv_write_kernel<float><<<T, 256, 0, stream>>>((float*)qkv, (const int32_t*)positions, (const float*)cos_t,
                                                           (const float*)sin_t, (const int32_t*)slot_mapping,
                                                           (float*)kpool, (float*)vpool, H, KVH, hd, rot, page_size);
    else
        rope_kv_write_kernel<bf16_t><<<T, 256, 0, stream>>>((bf16_t*)qkv, (const int32_t*)positions,
                                                            (const float*)cos_t, (const float*)sin_t,
                                                            (const int32_t*)slot_mapping, (bf16_t*)kpool,
                                                            (bf16_t*)vpool, H, KVH, hd, rot, page_size);
    return NI_LAUNCH_RESULT();
}

// parts: float32 [shares][T][(H + 2 KVH) * hd]; q [T, H * hd] and the pools in `dtype`
NI_EXPORT int ni_rope_kv_write_shares(const void* parts, int shares, void* q, const void* positions, const void* cos_t, const void* sin_t,
                                      const void* slot_mapping, void* kpool, void* vpool, int T, int H, int KVH, int hd, int rot, int page_size, int dtype,
                                      hipStream_t stream) {
    if (T <= 0 || shares < 1 || H <= 0 || KVH <= 0 || hd <= 0 || hd % 4 || rot < 0 || rot > hd || rot % 8 || page_size <= 0 || (rot && (!cos_t || !sin_t)) ||
        (slot_mapping && (!kpool || !vpool)) || !aligned_to(16, parts, q, cos_t) || !aligned_to(16, sin_t, kpool, vpool))
        return static_cast<int>(hipErrorInvalidValue);
    auto launch = [&](auto kernel, auto* qt, auto* kp, auto* vp) {
        kernel<<<T, 256, 0, stream>>>((const float*)parts, shares, qt, (const int32_t*)positions, (const float*)cos_t, (const float*)sin_t,
                                      (const int32_t*)slot_mapping, kp, vp, H, KVH, hd, rot, page_size);
    };
    auto typed = [&](auto* qt, auto* kp, auto* vp) {
        using E = std::remove_pointer_t<decltype(qt)>;
        if (shares == 2) launch(rope_kv_write_shares_kernel<E, 2>, qt, kp, vp);
        else if (shares == 3) launch(rope_kv_write_shares_kernel<E, 3>, qt, kp, vp);
        else if (shares == 4) launch(rope_kv_write_shares_kernel<E, 4>, qt, kp, vp);
        else if (shares == 6) launch(rope_kv_write_shares_kernel<E, 6>, qt, kp, vp);
        else if (shares == 8) launch(rope_kv_write_shares_kernel<E, 8>, qt, kp, vp);
        else if (shares == 10) launch(rope_kv_write_shares_kernel<E, 10>, qt, kp, vp);
        else if (shares == 12) launch(rope_kv_write_shares_kernel<E, 12>, qt, kp, vp);
        else launch(rope_kv_write_shares_kernel<E, 0>, qt, kp, vp);
    };
    if (dtype == 0) typed((float*)q, (float*)kpool, (float*)vpool);
    else typed((bf16_t*)q, (bf16_t*)kpool, (bf16_t*)vpool);
    return NI_LAUNCH_RESULT();
}

// activation: 0 silu, 1 gelu (tanh)
NI_EXPORT int ni_swiglu(const void* gu, void* out, int T, int I, int activation, int dtype, hipStream_t stream) {
    size_t n = static_cast<size_t>(T) * I;
    if (n == 0) return 0;
    const GatedUnit unit = GatedUnit::of(activation);
    if (dtype == 0) {
        if (I % 4 == 0)
            swiglu_vec_kernel<float, 4><<<blocks_for(n / 4, 256), 256, 0, stream>>>((const float*)gu, (float*)out, I, n / 4, unit);
        else
            swiglu_kernel<float><<<blocks_for(n, 256), 256, 0, stream>>>((const float*)gu, (float*)out, I, n, unit);
    } else {
        if (I % 8 == 0)
            swiglu_vec_kernel<bf16_t, 8><<<blocks_for(n / 8, 256), 256, 0, stream>>>((const bf16_t*)gu, (bf16_t*)out, I, n / 8, unit);
        else
            swiglu_kernel<bf16_t><<<blocks_for(n, 256), 256, 0, stream>>>((const bf16_t*)gu, (bf16_t*)out, I, n, unit);
    }
    return NI_LAUNCH_RESULT();
}

// out[i] = mean + std * normal(key, start + i), i < count, in the output's type (see counter_normal).
NI_EXPORT int ni_random_normal(void* out, size_t count, uint64_t key, uint64_t start, float mean, float std, int dtype,
                               hipStream_t stream) {
    if (count == 0) return 0;
    const unsigned blocks = static_cast<unsigned>(std::min<size_t>((count + 255) / 256, 65536));
    if (dtype == 0)
        random_normal_kernel<float><<<blocks, 256, 0, stream>>>((float*)out, count, key, start, mean, std);
    else
        random_normal_kernel<bf16_t><<<blocks, 256, 0, stream>>>((bf16_t*)out, count, key, start, mean, std);
    return NI_LAUNCH_RESULT();
}
