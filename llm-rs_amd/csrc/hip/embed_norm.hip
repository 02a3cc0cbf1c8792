// Token embedding into the 32-bit residual stream, and RMSNorm out of it.
#include "common.h"

typedef float embed_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 embed_bf16x8 __attribute__((ext_vector_type(8)));

// Eight values of a 16-bit row as one 16-byte load, widened and scaled (rows of a multiple of 8 values, 16-byte aligned).
__device__ __forceinline__ void load8_scaled(const bf16* src, float scale, float (&v)[8]) {
    embed_bf16x8 raw = *(const embed_bf16x8*)src;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (float)raw[j] * scale;
}
__device__ __forceinline__ void store8(float* dst, const float (&v)[8]) {
    *(embed_f32x4*)dst = embed_f32x4{v[0], v[1], v[2], v[3]};
    *(embed_f32x4*)(dst + 4) = embed_f32x4{v[4], v[5], v[6], v[7]};
}
template <class T>
__device__ __forceinline__ bool rows_by_eights(const T* table, const float* out, int D) {
    return sizeof(T) == 2 && D % 8 == 0 && ((uintptr_t)table & 15) == 0 && ((uintptr_t)out & 15) == 0;
}

// out[t, :] = float(table[tokens[t], :]) * scale   (reference: embed_batch_*, shaders/ops.metal:878-915,
// which has no scale: 1 there and for every architecture that does not ask for one)
// ADD: out[t, :] += the same, in 32-bit (a stream that is shown its tokens' embeddings again).
// WAVES: a vector of the token's position is added, feature 2i the sine and 2i + 1 the cosine of positions[t] * rate i, in
// 32-bit.  A rate is the sum of two 32-bit numbers, rates[i] and a small rates[n_rates + i]: what the product of position
// and rate loses to rounding (thousands of turns leave few digits for the angle) is carried along and turns the result by
// that little more.
__device__ __forceinline__ void position_wave(float pos, float rate, float rate_rest, float& s, float& c) {
    float a = pos * rate;
    float rest = fmaf(pos, rate, -a) + pos * rate_rest;
    float s0, c0;
    sincosf(a, &s0, &c0);
    s = fmaf(rest, c0, s0);
    c = fmaf(-rest, s0, c0);
}
// COPIES: the same rows into `copies` streams, `copy_stride` numbers apart.
template <class T, bool ADD, bool WAVES, bool COPIES = false>
__global__ void embed_rows_kernel(float* __restrict__ out, const T* __restrict__ table,
                                  const int* __restrict__ tokens, int D, int V, float scale,
                                  const int* __restrict__ positions, const float* __restrict__ rates, int copies = 1, size_t copy_stride = 0) {
    int t = blockIdx.x;
    const float pos = WAVES ? (float)positions[t] : 0.0f;
    const int n_rates = (D + 1) / 2;
    int row = tokens[t];
    row = row < 0 ? 0 : (row >= V ? V - 1 : row);  // the host has checked ids; never read outside the table
    const T* src = table + (size_t)row * D;
    float* dst = out + (size_t)t * D;
    if constexpr (sizeof(T) == 2) {
        if (rows_by_eights(table, out, D)) {           // (the same in all threads)
            for (int d = threadIdx.x * 8; d < D; d += blockDim.x * 8) {
                float v[8];
                load8_scaled((const bf16*)src + d, scale, v);
                if constexpr (ADD) {
                    embed_f32x4 a = *(const embed_f32x4*)(dst + d), b = *(const embed_f32x4*)(dst + d + 4);
#pragma unroll
                    for (int j = 0; j < 4; ++j) { v[j] += a[j]; v[4 + j] += b[j]; }
                }
                if constexpr (WAVES) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float s, c;
                        position_wave(pos, rates[(d >> 1) + j], rates[n_rates + (d >> 1) + j], s, c);
                        v[2 * j] += s;
                        v[2 * j + 1] += c;
                    }
                }
                store8(dst + d, v);
                if constexpr (COPIES)
                    for (int c = 1; c < copies; ++c) store8(dst + c * copy_stride + d, v);
            }
            return;
        }
    }
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
        float v = (ADD ? dst[d] : 0.0f) + to_f32(src[d]) * scale;
        if constexpr (WAVES) {
            float s, c;
            position_wave(pos, rates[d >> 1], rates[n_rates + (d >> 1)], s, c);
            v += (d & 1) ? c : s;
        }
        dst[d] = v;
        if constexpr (COPIES)
            for (int c = 1; c < copies; ++c) dst[c * copy_stride + d] = v;
    }
}

// One block per row: ss = sum x^2 in 32-bit, inv = 1/sqrt(ss/D + eps),
// y = (x * inv) * w, one rounding to the output type.  The weight multiplies
// directly (no 1+w).  Reference: rms_norm_batch, shaders/ops.metal:970-1003.
// The sum's order depends on D and the block size only, never on the row or batch.
template <class T>
__global__ void rmsnorm_rows_kernel(T* __restrict__ out, const float* __restrict__ x,
                                    const float* __restrict__ w, const int* __restrict__ rows, int D, float eps) {
    __shared__ float partial[16];
    int r = rows ? rows[blockIdx.x] : blockIdx.x;
    const float* src = x + (size_t)r * D;
    float ss = 0.0f;
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
        float v = src[d];
        ss = fmaf(v, v, ss);
    }
    ss = wave_sum(ss);
    int wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) partial[wave] = ss;
    __syncthreads();
    float total = 0.0f;
    for (int i = 0; i < nwaves; ++i) total += partial[i];
    float inv = 1.0f / sqrtf(total / (float)D + eps);
    T* dst = out + (size_t)blockIdx.x * D;
    for (int d = threadIdx.x; d < D; d += blockDim.x) dst[d] = from_f32<T>(src[d] * inv * w[d]);
}

// The same with the row held in registers between the sum and the scaling: one trip to
// memory instead of two, which is most of the time of a call with a few rows.  D % 4 == 0,
// D <= 4 * V4 * blockDim.  The sum's order again depends on D and the block size only.
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <class T, int V4>
__global__ void rmsnorm_rows_reg_kernel(T* __restrict__ out, const float* __restrict__ x,
                                        const float* __restrict__ w, const int* __restrict__ rows, int D, float eps) {
    __shared__ float partial[16];
    int r = rows ? rows[blockIdx.x] : blockIdx.x;
    const f32x4* src = (const f32x4*)(x + (size_t)r * D);
    int n4 = D / 4;
    f32x4 v[V4], ww[V4];
    float ss = 0.0f;
    // the norm's weight is asked for together with the row: a second trip to memory after the
    // sum would cost a call with few rows as much again as the first
#pragma unroll
    for (int i = 0; i < V4; ++i) {
        int idx = i * blockDim.x + threadIdx.x;
        v[i] = idx < n4 ? src[idx] : f32x4{0.f, 0.f, 0.f, 0.f};
        ww[i] = idx < n4 ? ((const f32x4*)w)[idx] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int i = 0; i < V4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) ss = fmaf(v[i][j], v[i][j], ss);
    ss = wave_sum(ss);
    int wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
    if ((threadIdx.x & 63) == 0) partial[wave] = ss;
    __syncthreads();
    float total = 0.0f;
    for (int i = 0; i < nwaves; ++i) total += partial[i];
    float inv = 1.0f / sqrtf(total / (float)D + eps);
    T* dst = out + (size_t)blockIdx.x * D;
#pragma unroll
    for (int i = 0; i < V4; ++i) {
        int idx = i * blockDim.x + threadIdx.x;
        if (idx < n4) {
            if constexpr (sizeof(T) == 2) {       // four 16-bit results as one 8-byte store
                typedef T T4 __attribute__((ext_vector_type(4)));
                T4 o4;
#pragma unroll
                for (int j = 0; j < 4; ++j) o4[j] = from_f32<T>(v[i][j] * inv * ww[i][j]);
                *(T4*)(dst + idx * 4) = o4;
            } else {
                f32x4 o4;
#pragma unroll
                for (int j = 0; j < 4; ++j) o4[j] = v[i][j] * inv * ww[i][j];
                *(f32x4*)(dst + idx * 4) = o4;
            }
        }
    }
}

template <bool ADD, bool WAVES>
static int embed_rows(hipStream_t stream, int dtype, float* out, const void* table, const int* tokens, int n_tokens, int D, int V, float scale,
                      const int* positions = nullptr, const float* rates = nullptr) {
    LLMRS_REQUIRE(n_tokens >= 0 && D > 0 && V > 0, "embed_rows: bad sizes T=%d D=%d V=%d", n_tokens, D, V);
    if (n_tokens == 0) return 0;
    if (dtype == LLMRS_F32)
        embed_rows_kernel<float, ADD, WAVES><<<n_tokens, 256, 0, stream>>>(out, (const float*)table, tokens, D, V, scale, positions, rates);
    else if (dtype == LLMRS_BF16)
        embed_rows_kernel<bf16, ADD, WAVES><<<n_tokens, 256, 0, stream>>>(out, (const bf16*)table, tokens, D, V, scale, positions, rates);
    else
        return llmrs_fail("embed_rows: unknown dtype %d", dtype);
    LLMRS_LAUNCH_CHECK("embed_rows");
    return 0;
}
extern "C" int llmrs_embed_rows(hipStream_t stream, int dtype, float* out, const void* table, const int* tokens,
                                int n_tokens, int D, int V, float scale) {
    return embed_rows<false, false>(stream, dtype, out, table, tokens, n_tokens, D, V, scale);
}
// The same rows into each of n_streams streams of [n_tokens, D].  (4 rows of 2048 into four streams, us: rows and then copies of the first
// stream 3.2 + 2.4, and 1.3 between them; here 3.3.)
extern "C" int llmrs_embed_streams(hipStream_t stream, int dtype, float* out, int n_streams, const void* table, const int* tokens,
                                   int n_tokens, int D, int V, float scale) {
    LLMRS_REQUIRE(n_streams >= 1 && n_tokens >= 0 && D > 0 && V > 0, "embed_streams: bad sizes T=%d D=%d V=%d streams=%d", n_tokens, D, V, n_streams);
    LLMRS_REQUIRE(dtype == LLMRS_F32 || dtype == LLMRS_BF16, "embed_streams: unknown dtype %d", dtype);
    if (n_tokens == 0) return 0;
    const size_t stride = (size_t)n_tokens * D;
    if (dtype == LLMRS_F32) embed_rows_kernel<float, false, false, true><<<n_tokens, 256, 0, stream>>>(out, (const float*)table, tokens, D, V, scale, nullptr, nullptr, n_streams, stride);
    else embed_rows_kernel<bf16, false, false, true><<<n_tokens, 256, 0, stream>>>(out, (const bf16*)table, tokens, D, V, scale, nullptr, nullptr, n_streams, stride);
    LLMRS_LAUNCH_CHECK("embed_streams");
    return 0;
}
// out[t, :] += float(table[tokens[t], :]) * scale
extern "C" int llmrs_embed_rows_add(hipStream_t stream, int dtype, float* out, const void* table, const int* tokens,
                                    int n_tokens, int D, int V, float scale) {
    return embed_rows<true, false>(stream, dtype, out, table, tokens, n_tokens, D, V, scale);
}

// out[t, :] = float(table[tokens[t], :]) * scale + waves of positions[t] (see the kernel); rates: [2][(D + 1) / 2] 32-bit
extern "C" int llmrs_embed_rows_waves(hipStream_t stream, int dtype, float* out, const void* table, const int* tokens,
                                      int n_tokens, int D, int V, float scale, const int* positions, const float* rates) {
    LLMRS_REQUIRE(positions && rates, "embed_rows: the position vector needs positions and rates");
    return embed_rows<false, true>(stream, dtype, out, table, tokens, n_tokens, D, V, scale, positions, rates);
}

// A token table beside a second table whose row is chosen by the token and the one before it:
//   out[t, :] = float(table[tokens[t], :]) * scale + float(pairs[row, :])
//   row = (previous * mul_prev + tokens[t] * mul_cur) mod buckets; for a sequence's first token (position 0) row `buckets`,
//   the last of the buckets + 1
// The token before an entry's first one comes from the request's state, last[slot]; the entry's last token is left there.
// The block of an entry's first token does both, reading before it writes, so no other block touches that state.
// copy (row stride ldc, or null): the same rows in the activation type, for whoever needs the embedding again later.
struct EmbedPairs {
    int buckets;
    long mul_prev, mul_cur;
    const int* positions;
    const int* token_entry;
    const int* q_starts;
    const int* slots;
    int* last;                   // [slots] at last_stride
    long last_stride;
};
template <class T>
__global__ __launch_bounds__(256) void embed_pairs_kernel(float* __restrict__ out, const T* __restrict__ table, const T* __restrict__ pairs,
                                                          const int* __restrict__ tokens, int D, int V, float scale, T* __restrict__ copy,
                                                          int ldc, EmbedPairs a) {
    const int t = blockIdx.x;
    const int token = tokens[t], e = a.token_entry[t], first = a.q_starts[e];
    const bool starts = a.positions[t] == 0;
    int previous = 0;
    if (t > first) previous = tokens[t - 1];
    else {
        int* last = a.last + (size_t)a.slots[e] * a.last_stride;
        previous = *last;
        __syncthreads();                               // (the whole block: every thread has read it)
        if (threadIdx.x == 0) *last = tokens[a.q_starts[e + 1] - 1];
    }
    long pick = ((long)previous * a.mul_prev + (long)token * a.mul_cur) % a.buckets;
    if (pick < 0) pick += a.buckets;
    const int row = token < 0 ? 0 : (token >= V ? V - 1 : token);  // the host has checked ids; never read outside the table
    const T* src = table + (size_t)row * D;
    const T* add = pairs + (size_t)(starts ? a.buckets : (int)pick) * D;
    float* dst = out + (size_t)t * D;
    T* cp = copy ? copy + (size_t)t * ldc : nullptr;
    if constexpr (sizeof(T) == 2) {
        if (rows_by_eights(table, out, D) && ((uintptr_t)pairs & 15) == 0 && ((uintptr_t)copy & 15) == 0 && ldc % 8 == 0) {     // (the same in all threads)
            for (int d = threadIdx.x * 8; d < D; d += 256 * 8) {
                float v[8], w[8];
                load8_scaled((const bf16*)src + d, scale, v);
                load8_scaled((const bf16*)add + d, 1.0f, w);
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] += w[j];
                store8(dst + d, v);
                if (cp) {
                    embed_bf16x8 o;
#pragma unroll
                    for (int j = 0; j < 8; ++j) o[j] = (bf16)v[j];
                    *(embed_bf16x8*)((bf16*)cp + d) = o;
                }
            }
            return;
        }
    }
    for (int d = threadIdx.x; d < D; d += 256) {
        float v = to_f32(src[d]) * scale + to_f32(add[d]);
        dst[d] = v;
        if (cp) cp[d] = from_f32<T>(v);
    }
}

// table: [V, D], pairs: [buckets + 1, D], both and `copy` in `dtype`; out: [n_tokens, D] 32-bit.
extern "C" int llmrs_embed_pairs(hipStream_t stream, int dtype, float* out, const void* table, const void* pairs, const int* tokens, int n_tokens,
                                 int D, int V, float scale, int buckets, long mul_prev, long mul_cur, const int* positions, const int* token_entry,
                                 const int* q_starts, const int* slots, int* last, long last_stride, void* copy, int ldc) {
    LLMRS_REQUIRE(out && table && pairs && tokens && n_tokens >= 0 && D > 0 && V > 0 && buckets > 0, "embed_pairs: bad sizes T=%d D=%d V=%d buckets=%d", n_tokens, D, V, buckets);
    LLMRS_REQUIRE(positions && token_entry && q_starts && slots && last && last_stride >= 1, "embed_pairs: the step's entries and the requests' last tokens are needed");
    LLMRS_REQUIRE(!copy || ldc >= D, "embed_pairs: the copy's rows are too short");
    if (n_tokens == 0) return 0;
    EmbedPairs a{buckets, mul_prev, mul_cur, positions, token_entry, q_starts, slots, last, last_stride};
    if (dtype == LLMRS_F32)
        embed_pairs_kernel<float><<<n_tokens, 256, 0, stream>>>(out, (const float*)table, (const float*)pairs, tokens, D, V, scale, (float*)copy, ldc, a);
    else if (dtype == LLMRS_BF16)
        embed_pairs_kernel<bf16><<<n_tokens, 256, 0, stream>>>(out, (const bf16*)table, (const bf16*)pairs, tokens, D, V, scale, (bf16*)copy, ldc, a);
    else
        return llmrs_fail("embed_pairs: unknown dtype %d", dtype);
    LLMRS_LAUNCH_CHECK("embed_pairs");
    return 0;
}

// out[t, :D] = x[t, :D] in the activation type; x 32-bit, both with row strides.
template <class T>
__global__ void cast_rows_kernel(T* __restrict__ out, int ldo, const float* __restrict__ x, int ldx, int D) {
    for (int d = threadIdx.x; d < D; d += blockDim.x) out[(size_t)blockIdx.x * ldo + d] = from_f32<T>(x[(size_t)blockIdx.x * ldx + d]);
}
extern "C" int llmrs_cast_rows(hipStream_t stream, int dtype, void* out, int ldo, const float* x, int ldx, int n_rows, int D) {
    LLMRS_REQUIRE(out && x && n_rows >= 0 && D > 0 && ldo >= D && ldx >= D, "cast_rows: bad sizes");
    if (n_rows == 0) return 0;
    if (dtype == LLMRS_F32) cast_rows_kernel<float><<<n_rows, 256, 0, stream>>>((float*)out, ldo, x, ldx, D);
    else if (dtype == LLMRS_BF16) cast_rows_kernel<bf16><<<n_rows, 256, 0, stream>>>((bf16*)out, ldo, x, ldx, D);
    else return llmrs_fail("cast_rows: unknown dtype %d", dtype);
    LLMRS_LAUNCH_CHECK("cast_rows");
    return 0;
}

// The norm of a sublayer's result on its way into the stream, for sublayers that read the stream as it is: one block a row,
//   h[t, :] += y[t, :] / sqrt(mean(y^2) + eps) * w      (32-bit)
//   x[t, :] = the new h[t, :] in the activation type     (x null: not wanted; a 32-bit engine reads h itself)
//   y[t, :] = 0                                          (where the next sublayer will add its result)
// norm 0: h stays, only x and y are made (in front of the first sublayer).  HELD: the row in registers between the sum and
// the stores, four features a piece, everything asked for at once; HELD 0: any width, one feature at a time.
template <class T, int HELD>
__global__ __launch_bounds__(256) void post_norm_rows_kernel(float* __restrict__ h, float* __restrict__ y, const float* __restrict__ w,
                                                             T* __restrict__ x, int D, float eps, int norm) {
    __shared__ float partial[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float* hrow = h + (size_t)blockIdx.x * D;
    float* yrow = y + (size_t)blockIdx.x * D;
    T* xrow = x ? x + (size_t)blockIdx.x * D : nullptr;
    if constexpr (HELD > 0) {
        const int n4 = D / 4;
        const f32x4 none = {0.f, 0.f, 0.f, 0.f};
        f32x4 yv[HELD], hv[HELD], wv[HELD];
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < HELD; ++i) {
            int idx = i * 256 + threadIdx.x;
            bool in = idx < n4;
            yv[i] = in && norm ? ((const f32x4*)yrow)[idx] : none;
            hv[i] = in ? ((const f32x4*)hrow)[idx] : none;
            wv[i] = in && norm ? ((const f32x4*)w)[idx] : none;
        }
        float inv = 0.0f;
        if (norm) {                                   // (the same in all threads)
#pragma unroll
            for (int i = 0; i < HELD; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) ss = fmaf(yv[i][j], yv[i][j], ss);
            ss = wave_sum(ss);
            if (lane == 0) partial[wave] = ss;
            __syncthreads();
            inv = 1.0f / sqrtf((partial[0] + partial[1] + partial[2] + partial[3]) / (float)D + eps);
        }
#pragma unroll
        for (int i = 0; i < HELD; ++i) {
            int idx = i * 256 + threadIdx.x;
            if (idx >= n4) continue;
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = hv[i][j] + yv[i][j] * inv * wv[i][j];
            if (norm) ((f32x4*)hrow)[idx] = v;
            ((f32x4*)yrow)[idx] = none;
            if (xrow) {
                typedef T T4 __attribute__((ext_vector_type(4)));
                T4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = from_f32<T>(v[j]);
                *(T4*)(xrow + idx * 4) = o;
            }
        }
    } else {
        float inv = 0.0f;
        if (norm) {
            float ss = 0.0f;
            for (int d = threadIdx.x; d < D; d += 256) ss = fmaf(yrow[d], yrow[d], ss);
            ss = wave_sum(ss);
            if (lane == 0) partial[wave] = ss;
            __syncthreads();
            inv = 1.0f / sqrtf((partial[0] + partial[1] + partial[2] + partial[3]) / (float)D + eps);
        }
        for (int d = threadIdx.x; d < D; d += 256) {
            float v = hrow[d];
            if (norm) {
                v += yrow[d] * inv * w[d];
                hrow[d] = v;
            }
            yrow[d] = 0.0f;
            if (xrow) xrow[d] = from_f32<T>(v);
        }
    }
}

// weight null: no norm (norm 0 above); x null or in `dtype`.
extern "C" int llmrs_post_norm_rows(hipStream_t stream, int dtype, float* h, float* y, const float* weight, void* x, int n_rows, int D, float eps) {
    LLMRS_REQUIRE(h && y && n_rows >= 0 && D > 0, "post_norm: bad sizes rows=%d D=%d", n_rows, D);
    LLMRS_REQUIRE(!weight || eps > 0.0f, "post_norm: eps must be positive, got %g", eps);
    if (n_rows == 0) return 0;
    if (dtype != LLMRS_F32 && dtype != LLMRS_BF16) return llmrs_fail("post_norm: unknown dtype %d", dtype);
    bool pieces = D % 4 == 0 && D <= 4 * 256 * 8 && ((uintptr_t)h & 15) == 0 && ((uintptr_t)y & 15) == 0 && ((uintptr_t)weight & 15) == 0 && ((uintptr_t)x & 15) == 0;
    int held = !pieces ? 0 : D <= 4 * 256 ? 1 : D <= 4 * 256 * 2 ? 2 : D <= 4 * 256 * 4 ? 4 : 8;
#define POST(T, N) post_norm_rows_kernel<T, N><<<n_rows, 256, 0, stream>>>(h, y, weight, (T*)x, D, eps, weight != nullptr)
#define POST_BY_WIDTH(T) do { if (held == 0) POST(T, 0); else if (held == 1) POST(T, 1); else if (held == 2) POST(T, 2); else if (held == 4) POST(T, 4); else POST(T, 8); } while (0)
    if (dtype == LLMRS_F32) POST_BY_WIDTH(float); else POST_BY_WIDTH(bf16);
#undef POST_BY_WIDTH
#undef POST
    LLMRS_LAUNCH_CHECK("post_norm");
    return 0;
}

// rows == nullptr: row i of x -> row i of out; else row rows[i] of x -> row i of out.
extern "C" int llmrs_rmsnorm(hipStream_t stream, int dtype, void* out, const float* x, const float* weight,
                             const int* rows, int n_rows, int D, float eps) {
    LLMRS_REQUIRE(n_rows >= 0 && D > 0, "rmsnorm: bad sizes rows=%d D=%d", n_rows, D);
    LLMRS_REQUIRE(eps > 0.0f, "rmsnorm: eps must be positive, got %g", eps);
    if (n_rows == 0) return 0;
    if (dtype != LLMRS_F32 && dtype != LLMRS_BF16) return llmrs_fail("rmsnorm: unknown dtype %d", dtype);
    int threads = D > 4096 ? 1024 : 256;     // a row of up to 4096 fits the registers of four waves: fewer waves to start and to wait for
    bool in_registers = D % 4 == 0 && D <= 4 * 4 * threads && ((uintptr_t)x & 15) == 0 && ((uintptr_t)weight & 15) == 0 &&
                        ((uintptr_t)out & 15) == 0;
    if (in_registers && dtype == LLMRS_F32)
        rmsnorm_rows_reg_kernel<float, 4><<<n_rows, threads, 0, stream>>>((float*)out, x, weight, rows, D, eps);
    else if (in_registers)
        rmsnorm_rows_reg_kernel<bf16, 4><<<n_rows, threads, 0, stream>>>((bf16*)out, x, weight, rows, D, eps);
    else if (dtype == LLMRS_F32)
        rmsnorm_rows_kernel<float><<<n_rows, threads, 0, stream>>>((float*)out, x, weight, rows, D, eps);
    else
        rmsnorm_rows_kernel<bf16><<<n_rows, threads, 0, stream>>>((bf16*)out, x, weight, rows, D, eps);
    LLMRS_LAUNCH_CHECK("rmsnorm");
    return 0;
}
