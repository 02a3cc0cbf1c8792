// C[m, n] = sum_k A[m, k] * W[n, k]: activations times a weight stored [out, in].
// What happens to the sum is the epilogue.
#pragma once
#include "common.h"

enum LlmrsEpilogue {
    LLMRS_EPI_STORE = 0,      // out[m, n] = acc, in the activation type
    LLMRS_EPI_STORE_F32 = 1,  // out[m, n] = acc, 32-bit (logits)
    LLMRS_EPI_ACCUM_F32 = 2,  // out[m, n] += acc, 32-bit (the residual stream)
    LLMRS_EPI_SWIGLU = 3,     // rows of W are (gate_0, up_0, gate_1, up_1, ...):
                              // out[m, n/2] = silu(acc[m, n]) * acc[m, n+1] for even n, activation type
    LLMRS_EPI_QKV = 4,        // rows of W are q heads, k heads, v heads: rotate q and k (adjacent pairs),
                              // q to out, k and v straight into the paged cache (QkvEpilogue)
    LLMRS_EPI_GLU_CLAMP = 5,  // 5 + slot, slot < LLMRS_GLU_SLOTS: rows of W as for SWIGLU; with the slot's constants (GluClamp),
                              // g = min(acc[m, n], limit), u = clamp(acc[m, n+1], -limit, limit),
                              // out[m, n/2] = g * sigmoid(alpha * (g + cubic * g^3)) * (u + up_add), activation type
                              // (up_add 1, cubic 0: the clamped gated activation; limit infinite, up_add 0,
                              // alpha 2 sqrt(2 / pi), cubic 0.044715: gelu(g) u in the tanh form of gelu)
};

// The constants of the gated epilogue with constants lie in a table in device memory, a slot for each set of them that a
// model has (llmrs_glu_clamp_slot, called when a feed-forward takes its weights, writes a slot once and for all); the
// epilogue's number says which slot, so no kernel's argument list holds them and a recorded step finds them as any
// other does.  Each source file that includes this has the table for itself (the variable is static), and by including
// it puts it on the list that llmrs_glu_clamp_slot writes through: no file can read a table that nothing writes.
#define LLMRS_GLU_SLOTS 256
struct GluClamp {
    float limit, alpha, cubic, up_add;
};
static __device__ GluClamp llmrs_glu_clamp[LLMRS_GLU_SLOTS];
static __global__ void glu_clamp_store_kernel(int slot, GluClamp p) { llmrs_glu_clamp[slot] = p; }
struct GluClampTable {
    void (*store)(hipStream_t stream, int slot, GluClamp p);
    GluClampTable* next;
};
extern GluClampTable* llmrs_glu_clamp_tables;        // gemm_simple.hip
static void glu_clamp_store(hipStream_t stream, int slot, GluClamp p) { glu_clamp_store_kernel<<<1, 1, 0, stream>>>(slot, p); }
static GluClampTable llmrs_glu_clamp_table = {glu_clamp_store, nullptr};
static const bool llmrs_glu_clamp_listed = (llmrs_glu_clamp_table.next = llmrs_glu_clamp_tables, llmrs_glu_clamp_tables = &llmrs_glu_clamp_table, true);

__host__ __device__ __forceinline__ bool epi_gated(int epi) { return epi == LLMRS_EPI_SWIGLU || epi >= LLMRS_EPI_GLU_CLAMP; }
// act(gate, up) of the gated epilogues, on 32-bit sums
__device__ __forceinline__ float gated_act(int epi, float g, float u) {
    if (epi == LLMRS_EPI_SWIGLU) return silu_f32(g) * u;
    const GluClamp p = llmrs_glu_clamp[epi - LLMRS_EPI_GLU_CLAMP];
    g = fminf(g, p.limit);
    u = fminf(fmaxf(u, -p.limit), p.limit);
    return g / (1.0f + expf(-p.alpha * fmaf(p.cubic * g * g, g, g))) * (u + p.up_add);
}

// What the q/k/v epilogue needs beside the sums.
struct QkvEpilogue {
    const int* positions;     // [M]
    const int* slot_map;      // [M] page * page_size + slot
    const float* inv_freq;    // [rotary_dim / 2]
    void* k_cache;            // in the activation type, as the rows
    void* v_cache;
    int n_heads, n_kv_heads, head_dim, rotary_dim;
    int page_size, num_pages, write_kv;
};

// RMSNorm without a kernel of its own, for steps of up to 16 tokens.  The product that adds into the
// 32-bit stream (its last writer before a norm) also leaves, for the norm that follows,
//   y[m, n]     = h[m, n] * weight[n]                  the new row times the norm's weight, rounded once (to bfloat16; 32-bit stays)
//   sumsq[m, p] = sum of h[m, n]^2 over the 16 (for some shapes 8) features n of group p
// (NextNorm); the product that follows takes y as its rows and multiplies each of its 32-bit sums by
//   inv[m] = 1 / sqrt(sum_p sumsq[m, p] / K + eps)       (RowScale; the groups are added in a fixed order)
// before its epilogue.  x W^T with x = h inv weight is the same number as inv (h weight) W^T; what
// differs from the norm kernel's output is where the one rounding to the activation type falls (on h weight
// instead of on h inv weight), not how many there are.
// With more rows, a product whose sums are split over blocks (k ranges) has a kernel that adds the parts up, and
// that kernel sees whole rows: with eps > 0 it finishes the following norm itself,
//   y[m, n] = bfloat16(h[m, n] * inv[m] * weight[n])
// which any product takes as plain rows (sumsq is not used then).
struct NextNorm {
    float* sumsq;          // [M, llmrs_gemm_next_parts(M, N, K)]: a part per 16 features, or per 8 (not used with eps > 0)
    void* y;               // [M, N] in the activation type, row stride ldy; null: nothing is left
    int ldy;
    const float* weight;   // [N]
    float eps;             // > 0: the norm is finished here (llmrs_gemm_norms_whole), else left to the next product
};
struct RowScale {
    const float* sumsq;    // [M, nparts]; null: no scale
    int nparts;
    float eps;
};

template <class T>
__device__ __forceinline__ void epilogue_store(int epi, void* out, int ldc, int m, int n, float v) {
    if (epi == LLMRS_EPI_STORE) ((T*)out)[(size_t)m * ldc + n] = from_f32<T>(v);
    else if (epi == LLMRS_EPI_STORE_F32) ((float*)out)[(size_t)m * ldc + n] = v;
    else if (epi == LLMRS_EPI_ACCUM_F32) ((float*)out)[(size_t)m * ldc + n] += v;
}

// Up to 16 rows, in 32-bit up to 32 (gemm_few.hip; scale, next and the q/k/v epilogue for up to 16): 16-byte aligned rows, K % 8 == 0 (32-bit: K % 32 == 0), the caller's to check.  1, 0 where the q/k/v
// epilogue's shape or alignment is not the kernel's, -1 on error (a deferred norm that cannot be taken); a launch's own
// error is the caller's to ask for.
int llmrs_gemm_few_bf16(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi,
                        const QkvEpilogue* qkv, const RowScale* scale, const NextNorm* next);
int llmrs_gemm_few_f32(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi,
                       const QkvEpilogue* qkv, const RowScale* scale, const NextNorm* next);
bool llmrs_half_tile_blocks(int N, int whole, int cus);
// 32-bit products on the matrix cores, tiles (gemm_f32_tiles.hip).  K % 32 == 0 and 16-byte aligned rows: the caller's to check.
// 0, or -1 on error.
int llmrs_gemm_f32_tiles(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi);
// The product left as the parts of its sum over k, [parts][M][N] 32-bit in `workspace` (gemm_mfma.hip): the number of
// parts, 0 when this product would not be split (nothing launched), -1 on error.
int llmrs_gemm_bf16_split_parts(hipStream_t stream, const bf16* A, int lda, const bf16* W, int M, int N, int K,
                                void* workspace, size_t workspace_bytes);
// The 16-byte-load kernels on MFMA (gemm_mfma.hip).  Return 1 when they took the
// product, 0 when its shape or alignment is not theirs, -1 on error.
// workspace: device memory for the partial sums of products that split K over blocks (may be null).
// qkv: needed when epi is LLMRS_EPI_QKV; such a call is taken only by the kernels that fuse it.
// scale, next: see RowScale and NextNorm; both only where llmrs_gemm_defers_norm(M, N, K) holds (next: with
// LLMRS_EPI_ACCUM_F32 only), or next with eps where llmrs_gemm_norms_whole(M, N, K) holds.
int llmrs_gemm_bf16_mfma(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc,
                         int M, int N, int K, int epi, void* workspace, size_t workspace_bytes,
                         const QkvEpilogue* qkv = nullptr, const RowScale* scale = nullptr, const NextNorm* next = nullptr);
// Whether the product of this shape, in bfloat16 or in 32-bit, goes to the kernel that can scale its rows' sums and leave a NextNorm.
extern "C" int llmrs_gemm_defers_norm(int M, int N, int K);
extern "C" int llmrs_gemm_f32_defers_norm(int M, int N, int K);
// Whether a product of that kind with N features can leave a NextNorm (the rows left are stored four features at once, and the widest
// weights' blocks take more tiles than they have waves).
extern "C" int llmrs_gemm_leaves_norm(int N);
// Whether the q/k/v epilogue, which stores four consecutive features of a head at once, takes heads of this geometry.  A product
// whose norm was left to it has no other way to its caches: who leaves the norm to it asks first.
extern "C" int llmrs_qkv_by_fours(int head_dim, int rotary_dim);
// The parts per row of the sums of squares that such a product leaves (NextNorm): what the caller sizes sumsq by.
extern "C" int llmrs_gemm_next_parts(int M, int N, int K);
// Which tiles a product of more than 64 rows takes that is too small for the square large ones (gemm_mfma.hip).
extern "C" int llmrs_gemm_mid_plan(int M, int N, int K, int epi);
// Whether the bfloat16 product of this shape, adding into the stream and given the workspace that
// llmrs_gemm_workspace_floats asks for, can finish the following norm (NextNorm with eps): where its sums are added up, or in a launch of its own.
extern "C" int llmrs_gemm_norms_whole(int M, int N, int K);
