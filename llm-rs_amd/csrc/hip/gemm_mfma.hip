// bfloat16 products on the matrix cores, 32-bit accumulation.
//
// Two kernels, chosen by M (the number of tokens in the step); up to 16 rows go to gemm_few.hip:
//   M <= 64  many requests decoding.  K % 64 == 0: gemm_ring.h.  Other K "skinny": every
//            weight is read once, straight from memory into MFMA operands; a block owns 16 to
//            112 output features and its waves split K.
//   M  > 64  "tiled": prompts.  Tiles of 128x128, 256x128, 256x192 or 256x256 outputs, K
//            in steps of 64 through double-buffered LDS, v_mfma_f32_32x32x16_bf16; when
//            K % 64 == 0 the tiles are loaded straight into LDS (by waves that do nothing
//            else), or, by the four waves of the largest, through registers between their
//            MFMAs (v_mfma_f32_16x16x32_bf16).
// Both need K % 8 == 0 and 16-byte aligned rows (16-byte loads); otherwise the
// caller falls back to the plain kernel.
//
// The order in which an output's products are summed depends on K, N, the
// kernel and the parts that K is split into, never on the row's place in the
// batch or the tile it falls in.
// Replaces the reference's matvec_bf16_simd / gemm_bf16 (shaders/ops.metal:52-159,
// :1090-1143); unlike gemm_bf16 (:1107) the accumulator is 32-bit.
#include "gemm_ring.h"
#include "gemm_tile.h"

__device__ __forceinline__ bf16x8 load8(const bf16* p) { return *(const bf16x8*)p; }
__device__ __forceinline__ bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = (bf16)0.0f;
    return z;
}

// act(gate, up) of the gated epilogues with the same instructions; the constants of those that have any are read from their slot
// once, before the loops that finish a tile (gated_act_of), not value by value
struct GatedAct {
    int epi;
    float limit, alpha2, cubic, up_add;        // alpha2 = -alpha log2(e)
};
__device__ __forceinline__ GatedAct gated_act_of(int epi) {
    GatedAct a{epi, 0.0f, 0.0f, 0.0f, 0.0f};
    if (epi >= LLMRS_EPI_GLU_CLAMP) {
        const GluClamp p = llmrs_glu_clamp[epi - LLMRS_EPI_GLU_CLAMP];
        a.limit = p.limit;
        a.alpha2 = p.alpha * -1.44269504088896341f;
        a.cubic = p.cubic;
        a.up_add = p.up_add;
    }
    return a;
}
__device__ __forceinline__ float gated_act_fast(const GatedAct& a, float g, float u) {
    if (a.epi == LLMRS_EPI_SWIGLU) return silu_fast_f32(g) * u;
    g = fminf(g, a.limit);
    u = fminf(fmaxf(u, -a.limit), a.limit);
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(__builtin_fmaf(a.cubic * g * g, g, g) * a.alpha2)) * (u + a.up_add);
}

// ---------------------------------------------------------------------------
// skinny: C^T[n, m] = sum_k W[n, k] X[m, k]
//   A operand = W rows: lane l holds row n0 + l%16 (+16 per feature tile), 8 consecutive k
//   B operand = X rows: lane l holds token l%16 (+16 per token tile), the same 8 k
//   C: lane l holds token l%16 and features 4*(l/16) + r, r = 0..3
// A lane's 8 k-values of one MFMA may be any 8, as long as both operands take
// the same; of a block of 64 k, lane group g takes [8g, 8g+8) for one MFMA and
// [32+8g, 32+8g+8) for the next, so that each load instruction reads 64
// contiguous bytes of every row and the two together one 128-byte line.
// A block owns NT*16 features and MT*16 tokens; its NW waves take the 64-wide
// k-blocks in turn (wave w: w, w+NW, ...), U of them per round with all loads of
// a round issued before its first MFMA, and add their sums in wave order.
// With gridDim.y > 1 the k-blocks are shared out over that many blocks as well
// (contiguous ranges): each writes its 32-bit partial sums to `partial`
// [gridDim.y][M][N] and gemm_splitk_finish_kernel adds them in order and applies
// the epilogue.  That is for weights with few rows and many tokens (17..64),
// where blocks of 64 features are needed to keep the tokens' rows from being
// read too often, and would otherwise be too few to fill the device.
// (For rows that are no whole k-blocks, and few short ones; gemm_ring.h takes the others.)
// LAST < 16: the last of a block's feature tiles has only LAST features (a block of 24 features is a tile and a
// half): the rows beyond are never asked for (their lanes load nothing and multiply zeros), so a weight whose
// 32-feature blocks would be an uneven number of rounds of the device can be shared out evenly.
// ---------------------------------------------------------------------------
template <int MT, int NT, int NW, int U, int LAST = 16>
__global__ __launch_bounds__(NW * 64) void gemm_skinny_kernel(const bf16* __restrict__ A, int lda,
                                                              const bf16* __restrict__ W, void* __restrict__ out,
                                                              int ldc, int M, int N, int K, int epi,
                                                              float* __restrict__ partial, QkvEpilogue qe, int rot_feats) {
    extern __shared__ __attribute__((aligned(16))) unsigned char skinny_smem[];
    float* red = (float*)skinny_smem;          // [NW][MT][NT][4][64]
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int row = lane & 15, g = lane >> 4;
    constexpr int BF = (NT - 1) * 16 + LAST;       // features of a block
    static_assert(LAST == 16 || LAST == 8, "a whole last tile, or half of one");
    int n0 = blockIdx.x * BF;
    const bool last_asks = LAST == 16 || row < LAST;   // whether this lane's row of the last tile exists
    const bf16* wp[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wp[nt] = W + (size_t)min(n0 + nt * 16 + row, N - 1) * K;
    const bf16* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xp[mt] = A + (size_t)min(mt * 16 + row, M - 1) * lda;
    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};

    int full = K / 64;             // blocks of 64 k that need no bounds
    int nkb = (K + 63) / 64;
    int per = (nkb + gridDim.y - 1) / gridDim.y;
    int lo = blockIdx.y * per;
    int kb_hi = min(nkb, lo + per);                        // this block's k-blocks: [lo, kb_hi)
    int cnt = max(min(full, kb_hi) - lo, 0);               // the full ones among them
    // The block walks its full k-blocks starting at `rot` and wraps round: with rot_feats > 0,
    // neighbouring groups of rot_feats features are at different places of their rows at any
    // moment.  Rows are a multiple of the memory channels' interleave apart, so blocks in step
    // would all ask the same few channels at once.  The start depends on the features alone
    // (a block's features lie within one group), not on how many of them a block takes.
    int rot = (cnt > 0 && rot_feats > 0) ? (n0 / rot_feats) % cnt : 0;
    auto turn = [&](int j) { int x = j + rot; return lo + (x >= cnt ? x - cnt : x); };
    // out += sum: the old values of the tile this wave will finish are asked for now, so that
    // their trip to memory runs beside the weights' instead of after the sums are ready
    float old[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const bool old_ahead = epi == LLMRS_EPI_ACCUM_F32 && partial == nullptr && wave < MT * NT;
    if (old_ahead) {
        int m = (wave / NT) * 16 + row, n = n0 + (wave % NT) * 16 + 4 * g;
        if (m < M)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) old[r] = ((const float*)out)[(size_t)m * ldc + n + r];
    }
    int j = wave;
    for (; j + (U - 1) * NW < cnt; j += U * NW) {
        bf16x8 w[U][NT][2], x[U][MT][2];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int k = turn(j + u * NW) * 64 + g * 8;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                if (LAST == 16 || nt < NT - 1 || last_asks) { w[u][nt][0] = load8(wp[nt] + k); w[u][nt][1] = load8(wp[nt] + k + 32); }
                else { w[u][nt][0] = zero8(); w[u][nt][1] = zero8(); }
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) { x[u][mt][0] = load8(xp[mt] + k); x[u][mt][1] = load8(xp[mt] + k + 32); }
        }
        __builtin_amdgcn_sched_barrier(0);   // keep the round's loads together, ahead of its MFMAs
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][nt][0], x[u][mt][0], acc[mt][nt], 0, 0, 0);
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][nt][1], x[u][mt][1], acc[mt][nt], 0, 0, 0);
                }
    }
    // what is left of this wave's turns, then the partial block if it is the wave's turn
    for (;; j += NW) {
        bool partial_turn = j == cnt && kb_hi > lo + cnt;   // one k-block past the full ones, cut by K
        if (j >= cnt && !partial_turn) break;
        int k = (partial_turn ? lo + cnt : turn(j)) * 64 + g * 8;
        bool v0 = k < K, v1 = k + 32 < K;
        bf16x8 w0[NT], w1[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            bool asks = LAST == 16 || nt < NT - 1 || last_asks;
            w0[nt] = v0 && asks ? load8(wp[nt] + k) : zero8();
            w1[nt] = v1 && asks ? load8(wp[nt] + k + 32) : zero8();
        }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            bf16x8 x0 = load8(xp[mt] + (v0 ? k : 0)), x1 = load8(xp[mt] + (v1 ? k + 32 : 0));
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[nt], x0, acc[mt][nt], 0, 0, 0);
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[nt], x1, acc[mt][nt], 0, 0, 0);
            }
        }
        if (partial_turn) break;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[(((wave * MT + mt) * NT + nt) * 4 + r) * 64 + lane] = acc[mt][nt][r];
    __syncthreads();
    // the (mt, nt) tiles are shared out over the waves; each is summed over the waves in order
    for (int tile = wave; tile < MT * NT; tile += NW) {
        int mt = tile / NT, nt = tile % NT;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float s = 0.0f;
#pragma unroll
            for (int w = 0; w < NW; ++w) s += red[(((w * MT + mt) * NT + nt) * 4 + r) * 64 + lane];
            v[r] = s;
        }
        int m = mt * 16 + row;
        int n = n0 + nt * 16 + 4 * g;
        if (m >= M) continue;
        if (LAST < 16 && nt == NT - 1 && 4 * g >= LAST) continue;     // the half of the last tile that is the next block's
        if (partial != nullptr) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) partial[((size_t)blockIdx.y * M + m) * N + n + r] = v[r];
        } else if (epi_gated(epi)) {
#pragma unroll
            for (int r = 0; r < 4; r += 2)
                if (n + r + 1 < N) ((bf16*)out)[(size_t)m * ldc + (n + r) / 2] = (bf16)gated_act(epi, v[r], v[r + 1]);
        } else if (epi == LLMRS_EPI_QKV) {
            if (n < N) store_qkv4<bf16>(qe, out, ldc, m, n, v);
        } else if (old_ahead && tile == wave) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) ((float*)out)[(size_t)m * ldc + n + r] = old[r] + v[r];
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) epilogue_store<bf16>(epi, out, ldc, m, n + r, v[r]);
        }
    }
}

// Adds the partial sums of a split product in order and applies the epilogue.
// One thread for two adjacent features (a gate/up pair when the epilogue is SwiGLU).
__global__ void gemm_splitk_finish_kernel(const float* __restrict__ partial, int splits, void* __restrict__ out,
                                          int ldc, int M, int N, int epi) {
    size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t pairs = (size_t)M * ((N + 1) / 2);
    if (idx >= pairs) return;
    int m = (int)(idx / ((N + 1) / 2)), n = 2 * (int)(idx % ((N + 1) / 2));
    float v0 = 0.0f, v1 = 0.0f;
    bool has1 = n + 1 < N;
    for (int s = 0; s < splits; ++s) {
        const float* p = partial + ((size_t)s * M + m) * N + n;
        v0 += p[0];
        if (has1) v1 += p[1];
    }
    if (epi_gated(epi)) {
        if (has1) ((bf16*)out)[(size_t)m * ldc + n / 2] = (bf16)gated_act(epi, v0, v1);
    } else {
        epilogue_store<bf16>(epi, out, ldc, m, n, v0);
        if (has1) epilogue_store<bf16>(epi, out, ldc, m, n + 1, v1);
    }
}

// The same for a product that adds into the 32-bit stream and is followed by a norm x / rms(x) * weight: a block
// for each row adds the parts in the same order, writes the stream's new row, and, having the whole row, the
// normed row as well (NextNorm with eps): no norm kernel runs.  Up to 16384 features (16 per thread), a multiple of 4.
__global__ __launch_bounds__(1024) void gemm_splitk_finish_norm_kernel(const float* __restrict__ partial, int splits,
                                                                        float* __restrict__ out, int ldc, int M, int N,
                                                                        NextNorm nn) {
    __shared__ float red[16];
    int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
    const float* p0 = partial + (size_t)m * N;
    float* o = out + (size_t)m * ldc;
    f32x4 h[4];
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int n = (i * (int)blockDim.x + tid) * 4;
        h[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (n < N) {
            f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int s = 0; s < splits; ++s) v += *(const f32x4*)(p0 + (size_t)s * M * N + n);
            h[i] = *(const f32x4*)(o + n) + v;
            *(f32x4*)(o + n) = h[i];
#pragma unroll
            for (int r = 0; r < 4; ++r) ss = fmaf(h[i][r], h[i][r], ss);
        }
    }
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    float total = 0.0f;
    for (int w = 0; w < waves; ++w) total += red[w];
    float inv = 1.0f / sqrtf(total / (float)N + nn.eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int n = (i * (int)blockDim.x + tid) * 4;
        if (n < N) {
            f32x4 w = *(const f32x4*)(nn.weight + n);
            bf16x4 y;
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = (bf16)(h[i][r] * inv * w[r]);
            *(bf16x4*)((bf16*)nn.y + (size_t)m * nn.ldy + n) = y;
        }
    }
}
// The norm alone, of rows that a product has added to as a whole: bound by reading them (2048 rows of 4096: 50 MB).  A block for each row, four pieces of it
// and of the weight asked for at once by every thread, 256 threads for 4096 features: 8.8 us, of 2048 features 5.9; the kernel above with no parts,
// 1024 threads that wait for the row before they ask for the weight, 12.2 and 6.9.  Features as there.
__global__ __launch_bounds__(1024) void norm_rows_kernel(const float* __restrict__ x, int ldx, int N, NextNorm nn) {
    __shared__ float red[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
    const float* row = x + (size_t)blockIdx.x * ldx;
    f32x4 h[4], w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = (i * (int)blockDim.x + tid) * 4;
        h[i] = n < N ? *(const f32x4*)(row + n) : f32x4{0.f, 0.f, 0.f, 0.f};
        w[i] = n < N ? *(const f32x4*)(nn.weight + n) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) ss = fmaf(h[i][r], h[i][r], ss);
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    float total = 0.0f;
    for (int i = 0; i < waves; ++i) total += red[i];
    const float inv = 1.0f / sqrtf(total / (float)N + nn.eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = (i * (int)blockDim.x + tid) * 4;
        if (n >= N) continue;
        bf16x4 y;
#pragma unroll
        for (int r = 0; r < 4; ++r) y[r] = (bf16)(h[i][r] * inv * w[i][r]);
        *(bf16x4*)((bf16*)nn.y + (size_t)blockIdx.x * nn.ldy + n) = y;
    }
}
static void launch_norm_rows(hipStream_t stream, const void* x, int ldx, int M, int N, const NextNorm& next) {
    norm_rows_kernel<<<M, min(1024, max(64, ceil_div(ceil_div(N, 16), 64) * 64)), 0, stream>>>((const float*)x, ldx, N, next);
}
// Adds the parts of a split product up: with the norm that follows where one is to be finished (NextNorm with eps).
static void launch_splitk_finish(hipStream_t stream, const float* partial, int splits, void* out, int ldc, int M, int N,
                                 int epi, const NextNorm* next) {
    if (next != nullptr && next->eps > 0.0f) {
        int threads = min(1024, ceil_div(ceil_div(N, 4), 64) * 64);
        gemm_splitk_finish_norm_kernel<<<M, threads, 0, stream>>>(partial, splits, (float*)out, ldc, M, N, *next);
        return;
    }
    size_t pairs = (size_t)M * ((N + 1) / 2);
    gemm_splitk_finish_kernel<<<ceil_div(pairs, 256), 256, 0, stream>>>(partial, splits, out, ldc, M, N, epi);
}

template <int MT, int NT, int NW, int U, int LAST = 16>
static void launch_skinny(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc,
                          int M, int N, int K, int epi, const QkvEpilogue* qkv, int splits = 1, float* partial = nullptr, int rot_feats = 0,
                          const NextNorm* next = nullptr) {
    size_t bytes = (size_t)NW * MT * NT * 4 * 64 * sizeof(float);
    static bool configured = false;
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)gemm_skinny_kernel<MT, NT, NW, U, LAST>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        configured = true;
    }
    gemm_skinny_kernel<MT, NT, NW, U, LAST><<<dim3(ceil_div(N, (NT - 1) * 16 + LAST), splits), NW * 64, bytes, stream>>>(
        A, lda, W, out, ldc, M, N, K, epi, splits > 1 ? partial : nullptr, qkv ? *qkv : QkvEpilogue{}, rot_feats);
    if (splits > 1) launch_splitk_finish(stream, partial, splits, out, ldc, M, N, epi, next);
}

// Stages: what fits in half of a unit's LDS, three to twelve.  (All of it, twice as many on their way, is no faster where a
// unit has one block, 64 rows of 28672 x 4096 46.6 against 46.0 us, and keeps a second block off where there are more, 16384 x 2048
// 20.4 against 19.2.)
template <int MT, int NT, int LAST, int KSUB>
constexpr int ring_stages() {
    constexpr int room = 75 * 1024 / ring_stage_bytes<MT, NT, LAST>(KSUB);
    return room > 12 ? 12 : room;
}
template <int MT, int NT, int LAST, int KSUB>
static void launch_ring(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi,
                        const QkvEpilogue* qkv, int splits = 1, float* partial = nullptr, int rot_feats = 0, const NextNorm* next = nullptr) {
    constexpr int STAGES = ring_stages<MT, NT, LAST, KSUB>();
    constexpr size_t bytes = (size_t)STAGES * ring_stage_bytes<MT, NT, LAST>(KSUB);
    static bool configured = false;
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)gemm_ring_kernel<MT, NT, LAST, KSUB, STAGES>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        configured = true;
    }
    gemm_ring_kernel<MT, NT, LAST, KSUB, STAGES><<<dim3(ceil_div(N, (NT - 1) * 16 + LAST), splits), 64 * ring_waves<MT>(), bytes, stream>>>(
        A, W, out, lda, ldc, M, N, K, epi, splits > 1 ? partial : nullptr, rot_feats, qkv ? *qkv : QkvEpilogue{});
    if (splits > 1) launch_splitk_finish(stream, partial, splits, out, ldc, M, N, epi, next);
}

// ---------------------------------------------------------------------------
// tiled: C[m, n] = sum_k X[m, k] W[n, k]
//   A operand = X rows (lane l: row l%32, k-chunk l/32), B operand = W rows
//   C: lane l holds feature l%32 and tokens 8*(r/4) + 4*(l/32) + r%4, r = 0..15,
//   so a store instruction writes 32 consecutive features of a token.
// ---------------------------------------------------------------------------
// BM x BN output tile per block of four waves (2 x 2); K in steps of BKT through
// two LDS buffers.  The global loads of the next P tiles are in flight, in
// registers, while this one is multiplied (one tile's product is far shorter than
// a trip to memory); the oldest of them is written to the other LDS buffer
// before the step's one barrier.
// LDS rows are padded by 16 bytes so that 16 lanes' 16-byte reads hit distinct banks.
template <int BM, int BN, int BKT, int P>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(const bf16* __restrict__ A, int lda,
                                                         const bf16* __restrict__ W, void* __restrict__ out,
                                                         int ldc, int M, int N, int K, int epi) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
    bf16* smem = (bf16*)smem_raw;
    constexpr int LDT = BKT + 8;
    constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 32, FN = TN / 32;
    constexpr int TPR = BKT / 8;              // threads that stage one row (16 bytes each)
    constexpr int RPP = 256 / TPR;            // rows staged per pass
    constexpr int A_IT = BM / RPP, W_IT = BN / RPP, BUF = (BM + BN) * LDT;
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int wm = wave >> 1, wn = wave & 1;
    int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    int srow = tid / TPR, schunk = (tid % TPR) * 8;
    bf16x8 ra[P][A_IT], rw[P][W_IT];     // ring of tiles in flight: slot t % P holds tile t

    auto load_tile = [&](int kt, int slot) {
        int k = kt * BKT + schunk;
        bool in = k < K;
#pragma unroll
        for (int i = 0; i < A_IT; ++i) {
            int gm = min(m0 + srow + RPP * i, M - 1);
            ra[slot][i] = in ? load8(A + (size_t)gm * lda + k) : zero8();
        }
#pragma unroll
        for (int i = 0; i < W_IT; ++i) {
            int gn = min(n0 + srow + RPP * i, N - 1);
            rw[slot][i] = in ? load8(W + (size_t)gn * K + k) : zero8();
        }
    };
    auto store_tile = [&](int buf, int slot) {
        bf16* as = smem + buf * BUF;
        bf16* ws = as + BM * LDT;
#pragma unroll
        for (int i = 0; i < A_IT; ++i) *(bf16x8*)(as + (srow + RPP * i) * LDT + schunk) = ra[slot][i];
#pragma unroll
        for (int i = 0; i < W_IT; ++i) *(bf16x8*)(ws + (srow + RPP * i) * LDT + schunk) = rw[slot][i];
    };

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    int nk = (K + BKT - 1) / BKT;
    load_tile(0, 0);
    store_tile(0, 0);
#pragma unroll
    for (int p = 1; p <= P - 1; ++p)
        if (p < nk) load_tile(p, p % P);
    __syncthreads();
    int frow = lane & 31, fk = (lane >> 5) * 8;
    for (int kt0 = 0; kt0 < nk; kt0 += P) {
#pragma unroll
        for (int p = 0; p < P; ++p) {            // unrolled so that ring slots are compile-time
            int kt = kt0 + p;
            if (kt >= nk) break;
            int cur = kt & 1;
            // tile kt's slot (p) is free: tile kt went to LDS in the step before
            if (kt + P < nk) load_tile(kt + P, p);
            const bf16* as = smem + cur * BUF + (wm * TM + frow) * LDT + fk;
            const bf16* ws = smem + cur * BUF + BM * LDT + (wn * TN + frow) * LDT + fk;
#pragma unroll
            for (int ks = 0; ks < BKT / 16; ++ks) {
                bf16x8 a[FM], b[FN];
#pragma unroll
                for (int i = 0; i < FM; ++i) a[i] = *(const bf16x8*)(as + i * 32 * LDT + ks * 16);
#pragma unroll
                for (int j = 0; j < FN; ++j) b[j] = *(const bf16x8*)(ws + j * 32 * LDT + ks * 16);
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
            }
            if (kt + 1 < nk) store_tile(cur ^ 1, (p + 1) % P);
            // (a bare barrier: __syncthreads() would wait for the later tiles' loads as well)
            block_sync_lds();
        }
    }

    // The accumulators must be indexed by constants or they end up in scratch memory:
    // the tiles are walked by a compile-time loop.
    static_for<0, FM * FN>([&](auto idx) {
        constexpr int i = decltype(idx)::value / FN, j = decltype(idx)::value % FN;
        int n = n0 + wn * TN + j * 32 + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            int m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            float v = acc[i][j][r];
            if (epi_gated(epi)) {
                float other = __shfl_xor(v, 1, 64);   // even lane: gate here, up next door
                if (!(lane & 1) && m < M && n + 1 < N)
                    ((bf16*)out)[(size_t)m * ldc + n / 2] = (bf16)gated_act(epi, v, other);
            } else if (m < M && n < N) {
                epilogue_store<bf16>(epi, out, ldc, m, n, v);
            }
        }
    });
}

template <int BM, int BN, int BKT, int P>
static int launch_tiled(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc,
                        int M, int N, int K, int epi) {
    static bool configured = false;
    size_t bytes = 2 * (BM + BN) * (BKT + 8) * sizeof(bf16);
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_tiled_kernel<BM, BN, BKT, P>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return llmrs_fail("gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        configured = true;
    }
    dim3 grid(ceil_div(N, BN), ceil_div(M, BM));
    if (grid.y > 65535) return llmrs_fail("gemm: M=%d is too large for one launch", M);
    gemm_tiled_kernel<BM, BN, BKT, P><<<grid, 256, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi);
    return 0;
}

// What a block of the tiled kernels does with its sums.  `smem` is the block's LDS (SMEM_BYTES of
// it), free once every wave has left the tile loop.
template <int BM, int BN, int WGM, int WGN, int SMEM_BYTES>
__device__ __forceinline__ void tile_epilogue(f32x16 (&acc)[BM / WGM / 32][BN / WGN / 32], unsigned char* smem,
                                              void* __restrict__ out, int ldc, int M, int N, int epi,
                                              float* __restrict__ partial, int m0, int n0) {
    constexpr int WAVES = WGM * WGN;
    constexpr int TM = BM / WGM, TN = BN / WGN, FM = TM / 32, FN = TN / 32;
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int wm = wave / WGN, wn = wave % WGN;
    if (partial != nullptr) {       // one part of the sum: as it is, for the kernel that adds the parts
        float* part = partial + (size_t)blockIdx.z * M * N;
        static_for<0, FM * FN>([&](auto idx) {
            constexpr int i = decltype(idx)::value / FN, j = decltype(idx)::value % FN;
            int n = n0 + wn * TN + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                int m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m < M && n < N) part[(size_t)m * N + n] = acc[i][j][r];
            }
        });
        return;
    }
    if (epi == LLMRS_EPI_ACCUM_F32) {
        // out += acc: a row block's old values are all asked for before the first sum is stored
        // (left to itself the compiler waits for each load before the store that follows it,
        // a trip to memory per value).
        float* o = (float*)out;
        static_for<0, FM>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            float old[FN][16];
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                int n = n0 + wn * TN + j * 32 + (lane & 31);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    int m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    old[j][r] = o[(size_t)min(m, M - 1) * ldc + min(n, N - 1)];
                }
            }
            static_for<0, FN>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                int n = n0 + wn * TN + j * 32 + (lane & 31);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    int m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (m < M && n < N) o[(size_t)m * ldc + n] = old[j][r] + acc[i][j][r];
                }
            });
        });
        return;
    }
    // 16-bit results: a lane holds one column of 16 rows, which stored as they lie would be 2 bytes
    // per lane and store.  The wave puts its tile through LDS (free after the loop's last barrier; each
    // wave has room for its own tile) and stores it row by row, 16 bytes per lane, whole lines at a time.
    bool staged = (epi == LLMRS_EPI_STORE || epi_gated(epi)) && ldc % 8 == 0 && ((uintptr_t)out & 15) == 0 &&
                  (epi_gated(epi) ? N % 16 == 0 : N % 8 == 0);
    if (staged) {
        const bool glu = epi_gated(epi);
        const GatedAct ga = gated_act_of(epi);
        const int cols = glu ? TN / 2 : TN;                       // columns of the wave's tile as stored
        const int row_bytes = cols * 2;
        static_assert(TN * 2 * TM * WAVES <= SMEM_BYTES, "the waves' tiles must fit in the tile buffers");
        unsigned char* mine = smem + wave * (TN * 2 * TM);
        // A lane holds one column of 16 rows, its neighbour (lane ^ 1) the next column.  Registers r and r + 1
        // are two adjacent rows: the two lanes trade one value of each pair (one DPP move, no LDS), after which the
        // even lane has both columns of row r and the odd lane both of row r + 1.  For the gate/up epilogue those
        // are a gate and its up (each lane finishes one output of the pair, none idles); for a plain store two
        // neighbouring results, written with one 4-byte store.
        const bool odd = lane & 1;
        static_for<0, FM * FN>([&](auto idx) {
            constexpr int i = decltype(idx)::value / FN, j = decltype(idx)::value % FN;
            int c = j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                int row = i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3) + (odd ? 1 : 0);
                float v0 = acc[i][j][r], v1 = acc[i][j][r + 1];
                float got = swap_neighbours(odd ? v0 : v1);
                float left = odd ? got : v0, right = odd ? v1 : got;       // columns c & ~1 and c | 1 of `row`
                if (glu) *(bf16*)(mine + row * row_bytes + (c / 2) * 2) = (bf16)gated_act_fast(ga, left, right);
                else {
                    bf16x2 two;
                    two[0] = (bf16)left;
                    two[1] = (bf16)right;
                    *(bf16x2*)(mine + row * row_bytes + (c & ~1) * 2) = two;
                }
            }
        });
        __builtin_amdgcn_s_waitcnt(0xc07f);                       // lgkmcnt(0): the wave's own LDS writes are done
        int lanes_per_row = cols / 8, rows_per_pass = 64 / lanes_per_row;
        int lr = lane / lanes_per_row, lc = (lane % lanes_per_row) * 8;
        int n_out = (glu ? (n0 + wn * TN) / 2 : n0 + wn * TN) + lc, n_lim = glu ? N / 2 : N;
        for (int row = lr; row < TM; row += rows_per_pass) {
            int m = m0 + wm * TM + row;
            if (m < M && n_out < n_lim)                           // (n_lim is a multiple of 8: a lane's 8 columns are in or out together)
                *(bf16x8*)((bf16*)out + (size_t)m * ldc + n_out) = *(const bf16x8*)(mine + row * row_bytes + lc * 2);
        }
        return;
    }
    static_for<0, FM * FN>([&](auto idx) {
        constexpr int i = decltype(idx)::value / FN, j = decltype(idx)::value % FN;
        int n = n0 + wn * TN + j * 32 + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            int m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            float v = acc[i][j][r];
            if (epi_gated(epi)) {
                float other = __shfl_xor(v, 1, 64);
                if (!(lane & 1) && m < M && n + 1 < N)
                    ((bf16*)out)[(size_t)m * ldc + n / 2] = (bf16)gated_act(epi, v, other);
            } else if (m < M && n < N) {
                epilogue_store<bf16>(epi, out, ldc, m, n, v);
            }
        }
    });
}

// ---------------------------------------------------------------------------
// tiled, loads straight into LDS: for K % 64 == 0.
// global_load_lds_dwordx4 moves 16 bytes per lane from memory into LDS without
// passing through registers; the 64 lanes of an instruction fill 1 KB of LDS in
// lane order, which is 8 tile rows of 64 k.  Rows therefore lie 128 bytes apart,
// unpadded, and bank conflicts are avoided by a swizzle instead: the 16-byte
// chunk c of row r lies in slot c ^ ((r >> 1) & 7) of its row (each lane simply
// fetches the chunk that belongs in its slot), so the 16 lanes of an operand read,
// which want the same chunk of 16 consecutive rows, hit 16 different bank groups.
// STAGES tiles are in LDS; the loads of the tile STAGES-1 ahead are issued
// before this tile's products and waited for (s_waitcnt vmcnt) only as far as the
// next tile needs.  No staging registers, no LDS store instructions.
// ---------------------------------------------------------------------------
template <int BM, int BN, int WGM, int WGN, int STAGES>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_dma_kernel(const bf16* __restrict__ A, int lda,
                                                       const bf16* __restrict__ W, void* __restrict__ out,
                                                       int ldc, int M, int N, int K, int epi,
                                                       float* __restrict__ partial) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char dma_smem[];
    constexpr int WAVES = WGM * WGN;                              // waves of a block, as a WGM x WGN grid over the tile
    constexpr int TM = BM / WGM, TN = BN / WGN, FM = TM / 32, FN = TN / 32;
    constexpr int STAGE_BYTES = (BM + BN) * 128;
    constexpr int A_GROUPS = BM / 8 / WAVES, W_GROUPS = BN / 8 / WAVES;   // 8-row groups per wave
    constexpr int LOADS = A_GROUPS + W_GROUPS;                     // load instructions per wave per tile
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int wm = wave / WGN, wn = wave % WGN;
    int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    int lrow = lane >> 3, lslot = lane & 7;

    // this lane's part of a tile: for each of its row groups, the row's global address of the
    // chunk that belongs in the lane's slot
    const bf16* ga[A_GROUPS];
    const bf16* gw[W_GROUPS];
#pragma unroll
    for (int i = 0; i < A_GROUPS; ++i) {
        int row = (wave * A_GROUPS + i) * 8 + lrow;
        ga[i] = A + (size_t)min(m0 + row, M - 1) * lda + ((lslot ^ ((row >> 1) & 7)) * 8);
    }
#pragma unroll
    for (int i = 0; i < W_GROUPS; ++i) {
        int row = (wave * W_GROUPS + i) * 8 + lrow;
        gw[i] = W + (size_t)min(n0 + row, N - 1) * K + ((lslot ^ ((row >> 1) & 7)) * 8);
    }
    // With gridDim.z > 1 the k-tiles are shared out over that many blocks (contiguous ranges): each
    // writes its 32-bit sums to `partial` [gridDim.z][M][N] and gemm_splitk_finish_kernel adds them
    // in order and applies the epilogue.  That is for products with too few tiles to fill the device.
    int nk_all = K / 64, per_split = (nk_all + gridDim.z - 1) / gridDim.z;
    int kt_lo = blockIdx.z * per_split;
    int nk = max(0, min(nk_all, kt_lo + per_split) - kt_lo);       // this block's k-tiles: [kt_lo, kt_lo + nk)
    auto issue = [&](int kt, int stage) {
        kt += kt_lo;
        unsigned base = __builtin_amdgcn_readfirstlane(stage * STAGE_BYTES + wave * A_GROUPS * 1024);
#pragma unroll
        for (int i = 0; i < A_GROUPS; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(ga[i] + kt * 64),
                                             (__attribute__((address_space(3))) void*)(dma_smem + base + i * 1024), 16, 0, 0);
        unsigned wbase = __builtin_amdgcn_readfirstlane(stage * STAGE_BYTES + BM * 128 + wave * W_GROUPS * 1024);
#pragma unroll
        for (int i = 0; i < W_GROUPS; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(gw[i] + kt * 64),
                                             (__attribute__((address_space(3))) void*)(dma_smem + wbase + i * 1024), 16, 0, 0);
    };

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

#pragma unroll
    for (int p = 0; p < STAGES - 1; ++p)
        if (p < nk) issue(p, p);
    if (nk >= STAGES - 1) wait_vmcnt<(STAGES - 2) * LOADS>(); else wait_vmcnt<0>();
    __syncthreads();

    int frow = lane & 31, h = lane >> 5;
    for (int kt = 0; kt < nk; ++kt) {
        int stage = kt % STAGES;
        if (kt + STAGES - 1 < nk) issue(kt + STAGES - 1, (kt + STAGES - 1) % STAGES);
        const unsigned char* as = dma_smem + stage * STAGE_BYTES;
        const unsigned char* ws = as + BM * 128;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            bf16x8 a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                int row = wm * TM + i * 32 + frow;
                a[i] = *(const bf16x8*)(as + row * 128 + (((ks * 2 + h) ^ ((row >> 1) & 7)) * 16));
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                int row = wn * TN + j * 32 + frow;
                b[j] = *(const bf16x8*)(ws + row * 128 + (((ks * 2 + h) ^ ((row >> 1) & 7)) * 16));
            }
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        // the next tile must have landed before anybody reads it; later tiles may still be on their way
        // (a bare barrier: __syncthreads() would wait for every load in flight, the later tiles' too)
        if (kt + STAGES - 1 < nk) wait_vmcnt<(STAGES - 2) * LOADS>(); else wait_vmcnt<0>();
        block_sync_lds();
    }

    tile_epilogue<BM, BN, WGM, WGN, STAGES * STAGE_BYTES>(acc, dma_smem, out, ldc, M, N, epi, partial, m0, n0);
}

template <int BM, int BN, int WGM, int WGN, int STAGES>
static int launch_dma(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc,
                      int M, int N, int K, int epi, int splits = 1, float* partial = nullptr, const NextNorm* next = nullptr,
                      bool finish = true) {
    static bool configured = false;
    size_t bytes = (size_t)STAGES * (BM + BN) * 128;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_dma_kernel<BM, BN, WGM, WGN, STAGES>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return llmrs_fail("gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        configured = true;
    }
    dim3 grid(ceil_div(N, BN), ceil_div(M, BM), splits);
    if (grid.y > 65535) return llmrs_fail("gemm: M=%d is too large for one launch", M);
    gemm_dma_kernel<BM, BN, WGM, WGN, STAGES><<<grid, 64 * WGM * WGN, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi,
                                                                                      splits > 1 ? partial : nullptr);
    if (splits > 1 && finish) launch_splitk_finish(stream, partial, splits, out, ldc, M, N, epi, next);
    return 0;
}

// ---------------------------------------------------------------------------
// tiled, two groups of waves out of step: for K % 64 == 0, 256 x 256 tiles.
// In the tile loop above all eight waves of a block do the same thing at the same
// time: after each barrier every wave asks memory for the next tile, then reads LDS,
// then feeds the matrix cores, and the two waves that share a SIMD compete for each in
// turn.  Here the block's waves are two groups of four, one wave of each on every SIMD.
// A k-tile of 64 is four phases with a barrier after each: the operands of its first
// half from LDS into registers; their 16 MFMAs; the second half's operands; their
// MFMAs.  The second group runs one phase behind the first, so while one wave of a
// SIMD multiplies, the other reads LDS.  Both groups ask memory for the tile after the
// next in the same phase (the first group's first, the second group's fourth of the
// tile before), the first in which the buffer's last reader is done, and wait for it
// four phases later.  Every wave passes the same number of barriers.  Same LDS layout
// as above (two tiles, rows of 128 bytes, chunks swizzled), same order of sums: the
// results are bitwise those of the loop above.  A wave multiplies at raised priority.
// (Measured on MI355X, 2048 x 4096 times 24576 features: 2-5 % faster than the loop above when
// the product runs back to back with itself, 1 % inside a prompt step of the 8B shape.)
// ---------------------------------------------------------------------------
template <int BM, int BN, int WGM, int WGN, bool BUF = false>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_pingpong_kernel(const bf16* __restrict__ A, int lda,
                                                            const bf16* __restrict__ W, void* __restrict__ out,
                                                            int ldc, int M, int N, int K, int epi) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char pp_smem[];
    constexpr int WAVES = WGM * WGN;
    static_assert(WAVES == 8, "two groups of four waves");
    constexpr int TM = BM / WGM, TN = BN / WGN, FM = TM / 32, FN = TN / 32;
    constexpr int STAGE_BYTES = (BM + BN) * 128;
    constexpr int A_GROUPS = BM / 8 / WAVES, W_GROUPS = BN / 8 / WAVES;   // 8-row groups per wave
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int wm = wave / WGN, wn = wave % WGN;
    int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    int lrow = lane >> 3, lslot = lane & 7;
    const bf16* ga[A_GROUPS];
    const bf16* gw[W_GROUPS];
#pragma unroll
    for (int i = 0; i < A_GROUPS; ++i) {
        int row = (wave * A_GROUPS + i) * 8 + lrow;
        ga[i] = A + (size_t)min(m0 + row, M - 1) * lda + ((lslot ^ ((row >> 1) & 7)) * 8);
    }
#pragma unroll
    for (int i = 0; i < W_GROUPS; ++i) {
        int row = (wave * W_GROUPS + i) * 8 + lrow;
        gw[i] = W + (size_t)min(n0 + row, N - 1) * K + ((lslot ^ ((row >> 1) & 7)) * 8);
    }
    const int nk = K / 64;
    // BUF: the loads go through buffer descriptors (a scalar base and a 32-bit offset per lane)
    // instead of a 64-bit address per lane; the caller sees to it that both operands are under 4 GB.
    // (The descriptor type and builtins exist for the device only.)
#if defined(__HIP_DEVICE_COMPILE__)
    __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)min((size_t)M * lda * 2, (size_t)0xffffffffu), 0x00020000);
    __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)W, 0, (int)min((size_t)N * K * 2, (size_t)0xffffffffu), 0x00020000);
#endif
    unsigned oa[A_GROUPS], ow[W_GROUPS];
#pragma unroll
    for (int i = 0; i < A_GROUPS; ++i) oa[i] = (unsigned)((const char*)ga[i] - (const char*)A);
#pragma unroll
    for (int i = 0; i < W_GROUPS; ++i) ow[i] = (unsigned)((const char*)gw[i] - (const char*)W);
    auto issue = [&](int kt) {
        if (kt >= nk) return;
        int stage = kt & 1;
        unsigned base = __builtin_amdgcn_readfirstlane(stage * STAGE_BYTES + wave * A_GROUPS * 1024);
#pragma unroll
        for (int i = 0; i < A_GROUPS; ++i) {
#if defined(__HIP_DEVICE_COMPILE__)
            if constexpr (BUF)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(pp_smem + base + i * 1024), 16, oa[i], kt * 128, 0, 0);
            else
#endif
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(ga[i] + kt * 64),
                                                 (__attribute__((address_space(3))) void*)(pp_smem + base + i * 1024), 16, 0, 0);
        }
        unsigned wbase = __builtin_amdgcn_readfirstlane(stage * STAGE_BYTES + BM * 128 + wave * W_GROUPS * 1024);
#pragma unroll
        for (int i = 0; i < W_GROUPS; ++i) {
#if defined(__HIP_DEVICE_COMPILE__)
            if constexpr (BUF)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void*)(pp_smem + wbase + i * 1024), 16, ow[i], kt * 128, 0, 0);
            else
#endif
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(gw[i] + kt * 64),
                                                 (__attribute__((address_space(3))) void*)(pp_smem + wbase + i * 1024), 16, 0, 0);
        }
    };
    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    auto barrier = [] {
        __builtin_amdgcn_sched_barrier(0);
        block_sync_lds();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto lds_done = [] { __builtin_amdgcn_s_waitcnt(0xc07f); };     // lgkmcnt(0)
    int frow = lane & 31, h = lane >> 5;
    bf16x8 a[2][FM], b[2][FN];
    auto read_half = [&](int kt, int half) {
        const unsigned char* as = pp_smem + (kt & 1) * STAGE_BYTES;
        const unsigned char* ws = as + BM * 128;
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
            int ks = half * 2 + s2;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                int row = wm * TM + i * 32 + frow;
                a[s2][i] = *(const bf16x8*)(as + row * 128 + (((ks * 2 + h) ^ ((row >> 1) & 7)) * 16));
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                int row = wn * TN + j * 32 + frow;
                b[s2][j] = *(const bf16x8*)(ws + row * 128 + (((ks * 2 + h) ^ ((row >> 1) & 7)) * 16));
            }
        }
    };
    auto multiply = [&] {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s2][i], b[s2][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_s_setprio(0);
    };

    issue(0);
    wait_vmcnt<0>();
    barrier();
    const int grp = wave >> 2;
    // Phases as the whole block sees them, p = 0, 1, ...: the first group works on k-tile kt in
    // phases 4 kt .. 4 kt + 3, the second in 4 kt + 1 .. 4 kt + 4.  Tile kt + 1 goes into the buffer
    // of tile kt - 1, whose last reader (the second group's third phase) is done when phase 4 kt
    // begins; it is first read in phase 4 kt + 4.
    if (grp == 1) { issue(1); barrier(); }
    for (int kt = 0; kt < nk; ++kt) {
        read_half(kt, 0);
        if (grp == 0) issue(kt + 1);                     // phase 4 kt: the buffer of tile kt - 1 is free
        lds_done();
        barrier();
        multiply();
        barrier();
        read_half(kt, 1);
        lds_done();
        if (grp == 1) wait_vmcnt<0>();                   // its part of tile kt + 1 (asked for four phases ago)
        barrier();
        if (grp == 1) issue(kt + 2);                     // phase 4 kt + 4: the buffer of tile kt is free
        multiply();
        if (grp == 0) wait_vmcnt<0>();
        barrier();
    }
    if (grp == 0) barrier();
    tile_epilogue<BM, BN, WGM, WGN, 2 * STAGE_BYTES>(acc, pp_smem, out, ldc, M, N, epi, nullptr, m0, n0);
}

template <int BM, int BN, int WGM, int WGN, bool BUF = false>
static int launch_pingpong(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc,
                           int M, int N, int K, int epi) {
    static bool configured = false;
    size_t bytes = (size_t)2 * (BM + BN) * 128;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_pingpong_kernel<BM, BN, WGM, WGN, BUF>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return llmrs_fail("gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        configured = true;
    }
    dim3 grid(ceil_div(N, BN), ceil_div(M, BM));
    if (grid.y > 65535) return llmrs_fail("gemm: M=%d is too large for one launch", M);
    gemm_pingpong_kernel<BM, BN, WGM, WGN, BUF><<<grid, 64 * WGM * WGN, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi);
    return 0;
}

// ---------------------------------------------------------------------------
// tiled, four waves: for K % 64 == 0, tiles of 256 x 256, 256 x 192 and 256 x 128.
// One wave per SIMD with a tile of 128 x 128 outputs, all of them in the accumulation registers (256 of them):
// a third fewer LDS reads per MFMA than the eight-wave tiles, and nothing shares the SIMD with the wave, so the
// loop is written so that the wave itself always has work in flight.  A k-tile of 64 is four steps, half of its k times half of the
// wave's tokens each; a step asks LDS for operands of the next one, moves a quarter of the next k-tile from registers into the
// other LDS buffer, asks memory for the same quarter of the k-tile after that, and multiplies the operands
// asked for before.  Loads from memory pass through registers here, two k-tiles ahead of their use (the
// loads straight into LDS of the loops above hold a wave that has no partner on its SIMD up while the memory
// pipeline takes them).  The barrier between k-tiles stands before the last step's products, which run on
// registers read before it: the matrix cores work across it.  Same LDS layout as the loops above, and a sum's products are added in
// the order of k as there: bitwise the same results.  The epilogue is a template argument: with all of them in one kernel the
// compiler keeps a tile's 256 sums and every epilogue's temporaries alive together and spills.
// What bounds it: the clock, which follows the power that the matrix cores and LDS draw.  v_mfma_f32_16x16x32_bf16 with features as its rows (a lane
// then ends with four consecutive features of a token, so gated pairs need no neighbour and results go out by whole lines)
// against v_mfma_f32_32x32x16_bf16 with results stored from where they lay, us: 2048 rows 57344 x 8192 gated 1381 -> 1338 (1.44
// PFLOP/s), 8192 x 28672 added to 723 -> 697, 4096 x 14336 213 -> 206, 4096 x 4096 69.7 -> 64.8, 6144 x 4096 85.7 -> 82.1; 2032 rows
// 16384 x 2048 gated 113.5 -> 106.3; 571 rows 18112 x 128 added to 29.4 -> 19.3.  Found slower: grids of 6 x 24 tiles of 256 x 128
// with long rows that store or gate (1360 rows 3040 x 9152 gated 89.4 -> 93.4, 3040 x 4096 42.9 -> 45.1, 1536 rows 3072 x 9152 stored 90.8 -> 93.9), which
// neither their neighbours do (5 x 24 0.94-0.97 of the time, 6 x 26 and 6 x 28 0.98-1.0) nor the same grids adding to the stream (0.94-0.98).
// ---------------------------------------------------------------------------
// What a wave of the four-wave tile does with its sums.  acc[i][j] are 16 tokens x 16 features, and a lane holds four consecutive
// features of one token: a gated pair lies in one lane.  32-bit results leave by bands_to_f32; 16-bit ones likewise, a band of 32 tokens
// at a time, as whole rows of the band, 16 bytes a lane.
// epi: the epilogue's number as the caller gave it (EPI with its slot, where it has one)
template <int BM, int BN, int EPI>
__device__ __forceinline__ void band_epilogue(f32x4 (&acc)[BM / 32][BN / 32], unsigned char* smem, void* __restrict__ out,
                                              int ldc, int M, int N, int m0, int n0, int epi) {
    constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16;
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int wm = wave / 2, wn = wave % 2;
    if constexpr (EPI == LLMRS_EPI_ACCUM_F32 || EPI == LLMRS_EPI_STORE_F32) {
        bands_to_f32<FM, FN, false>(smem + wave * (16 * (TN * 4 + 16)), (float*)out, ldc, M, N, m0 + wm * TM, n0 + wn * TN, EPI == LLMRS_EPI_ACCUM_F32,
                                    [&](auto ic, auto jc) { return acc[decltype(ic)::value][decltype(jc)::value]; });
    } else {
        int token = lane & 15, four = (lane >> 4) * 4;
        constexpr bool glu = EPI == LLMRS_EPI_SWIGLU || EPI == LLMRS_EPI_GLU_CLAMP;
        const GatedAct ga = gated_act_of(EPI == LLMRS_EPI_GLU_CLAMP ? epi : EPI);
        constexpr int cols = glu ? TN / 2 : TN;      // columns of the wave's band as stored
        constexpr int row_bytes = cols * 2 + 16;
        unsigned char* mine = smem + wave * (32 * row_bytes);
        constexpr int pieces_per_row = cols / 8, PIECES = 32 * pieces_per_row / 64;     // 16-byte pieces: in a row of the band, of a lane
        static_assert(32 * pieces_per_row % 64 == 0, "a band is the same number of pieces for every lane");
        int n_first = glu ? (n0 + wn * TN) / 2 : n0 + wn * TN, n_lim = glu ? N / 2 : N;
        auto write = [&](auto bandc) {
            static_for<0, 2 * FN>([&](auto jc) {
                constexpr int half = decltype(jc)::value / FN, j = decltype(jc)::value % FN;
                f32x4 v = acc[2 * decltype(bandc)::value + half][j];
                unsigned char* at = mine + (half * 16 + token) * row_bytes;
                if constexpr (glu) {
                    bf16x2 two;
                    two[0] = (bf16)gated_act_fast(ga, v[0], v[1]);
                    two[1] = (bf16)gated_act_fast(ga, v[2], v[3]);
                    *(bf16x2*)(at + j * 16 + four) = two;
                } else {
                    bf16x4 o4;
#pragma unroll
                    for (int r = 0; r < 4; ++r) o4[r] = (bf16)v[r];
                    *(bf16x4*)(at + (j * 16 + four) * 2) = o4;
                }
            });
        };
        write(std::integral_constant<int, 0>{});
        static_for<0, FM / 2>([&](auto ic) {
            constexpr int band = decltype(ic)::value;
            bf16x8 v[PIECES];
            asm volatile("" ::: "memory");           // (a wave's LDS accesses are carried out in the order it asks for them)
#pragma unroll
            for (int p = 0; p < PIECES; ++p) {
                int piece = p * 64 + lane;
                v[p] = *(const bf16x8*)(mine + piece / pieces_per_row * row_bytes + piece % pieces_per_row * 16);
            }
            asm volatile("" ::: "memory");
            if constexpr (band + 1 < FM / 2) write(std::integral_constant<int, band + 1>{});
#pragma unroll
            for (int p = 0; p < PIECES; ++p) {
                int piece = p * 64 + lane, m = m0 + wm * TM + band * 32 + piece / pieces_per_row, lc = piece % pieces_per_row * 8;
                if (m < M && n_first + lc < n_lim)                // (n_lim is a multiple of 8: a lane's 8 columns are in or out together)
                    *(bf16x8*)((bf16*)out + (size_t)m * ldc + n_first + lc) = v[p];
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    }
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// A quarter of a wave's loads of a k-tile: of `groups` loads those from first_of(groups, q) up to first_of(groups, q + 1).
constexpr int first_of(int groups, int q) { return q * groups / 4; }
constexpr int quarter_of(int groups, int q) { return first_of(groups, q + 1) - first_of(groups, q); }

// TAIL: the `over` rows, up to 16, that follow the M whole tiles' rows.  A column of tiles has their 16 features of a wave's B operands in LDS
// anyway, so its waves share those features out: a wave multiplies 16 more features by 16 more tokens, one MFMA for 64,
// with the tokens straight from memory in the operand's layout, a k-tile ahead.  (A launch of their own reads the whole weight again:
// 2064 rows 57344 x 8192 gated 1548 -> 1400 us, 2048 rows 1346; 8192 x 28672 added to 789 -> 698, 8192 x 8192 252 -> 210; 8208 rows 28672 x 4096
// gated 1428 -> 1366.)
template <int EPI>
__device__ __forceinline__ void tail_epilogue(f32x4 v, void* __restrict__ out, int ldc, int N, int m, int n, int epi) {
    if constexpr (EPI == LLMRS_EPI_SWIGLU || EPI == LLMRS_EPI_GLU_CLAMP) {
        const GatedAct ga = gated_act_of(EPI == LLMRS_EPI_GLU_CLAMP ? epi : EPI);
        bf16* o = (bf16*)out + (size_t)m * ldc + n / 2;
        if (n + 1 < N) o[0] = (bf16)gated_act_fast(ga, v[0], v[1]);
        if (n + 3 < N) o[1] = (bf16)gated_act_fast(ga, v[2], v[3]);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < N) epilogue_store<bf16>(EPI, out, ldc, m, n + r, v[r]);
    }
}

template <int BM, int BN, int EPI, int TAIL>
__global__ __launch_bounds__(256) void gemm_fourwave_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W,
                                                            void* __restrict__ out, int ldc, int M, int N, int K, int epi, int over) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char fw_smem[];
    constexpr int WAVES = 4;
    constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16, FNH = (FN + 1) / 2;
    constexpr int STAGE_BYTES = (BM + BN) * 128;
    constexpr int A_GROUPS = BM / 8 / WAVES, W_GROUPS = BN / 8 / WAVES;   // 8-row groups per wave
    static_assert(BM == 256 && BN % 32 == 0 && FM * FN <= 64, "a wave's sums fill at most the 256 accumulation registers");
    static_assert(32 * (TN * 2 + 16) * WAVES <= STAGE_BYTES && 16 * (TN * 4 + 16) * WAVES <= STAGE_BYTES, "the waves' bands must fit in one of the tile buffers");
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int wm = wave / 2, wn = wave % 2;
    int tile_row, tile_column;
    tile_of_block(K, tile_row, tile_column);
    int m0 = tile_row * BM, n0 = tile_column * BN;
    int lrow = lane >> 3, lslot = lane & 7;
    // this lane's part of a tile: for each of its row groups, the byte offset of the chunk that belongs in the lane's
    // slot of the LDS image (the caller sees to it that both operands are under 4 GB: buffer descriptors)
    unsigned oa[A_GROUPS], ow[W_GROUPS];
#pragma unroll
    for (int i = 0; i < A_GROUPS; ++i) {
        int row = (wave * A_GROUPS + i) * 8 + lrow;
        oa[i] = (unsigned)(((size_t)min(m0 + row, M - 1) * lda + ((lslot ^ ((row >> 1) & 7)) * 8)) * 2);
    }
#pragma unroll
    for (int i = 0; i < W_GROUPS; ++i) {
        int row = (wave * W_GROUPS + i) * 8 + lrow;
        ow[i] = (unsigned)(((size_t)min(n0 + row, N - 1) * K + ((lslot ^ ((row >> 1) & 7)) * 8)) * 2);
    }
    const int nk = K / 64;
#if defined(__HIP_DEVICE_COMPILE__)
    __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)min((size_t)(M + (TAIL != 0 ? over : 0)) * lda * 2, (size_t)0xffffffffu), 0x00020000);
    __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)W, 0, (int)min((size_t)N * K * 2, (size_t)0xffffffffu), 0x00020000);
#endif
    u32x4 sa[A_GROUPS], sw_[W_GROUPS];          // the k-tile on its way, in registers
    // quarter q of this wave's loads of k-tile kt, into registers (past the end: the last tile once more, never used)
    auto ask = [&](int kt, auto qc) {
        constexpr int q = decltype(qc)::value;
        kt = min(kt, nk - 1);
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
        for (int i = first_of(A_GROUPS, q); i < first_of(A_GROUPS, q + 1); ++i) sa[i] = __builtin_amdgcn_raw_buffer_load_b128(ra, oa[i], kt * 128, 0);
#pragma unroll
        for (int i = first_of(W_GROUPS, q); i < first_of(W_GROUPS, q + 1); ++i) sw_[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, ow[i], kt * 128, 0);
#endif
    };
    // quarter q of the registers into the LDS buffer of k-tile kt: a load's 64 lanes fill 1 KB in lane order
    auto put = [&](int kt, auto qc) {
        constexpr int q = decltype(qc)::value;
        unsigned char* st = fw_smem + (kt & 1) * STAGE_BYTES;
#pragma unroll
        for (int i = first_of(A_GROUPS, q); i < first_of(A_GROUPS, q + 1); ++i) *(u32x4*)(st + (wave * A_GROUPS + i) * 1024 + lane * 16) = sa[i];
#pragma unroll
        for (int i = first_of(W_GROUPS, q); i < first_of(W_GROUPS, q + 1); ++i) *(u32x4*)(st + BM * 128 + (wave * W_GROUPS + i) * 1024 + lane * 16) = sw_[i];
    };
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int frow = lane & 15, h = lane >> 4;
    int sw = (frow >> 1) & 7;
    // LDS offsets of this lane's chunk for each half of a k-tile, 32 k long (row tiles lie 2 KB apart)
    unsigned offa[2], offb[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        unsigned chunk = (unsigned)(((ks * 4 + h) ^ sw) * 16);
        offa[ks] = (wm * TM + frow) * 128 + chunk;
        offb[ks] = BM * 128 + (wn * TN + frow) * 128 + chunk;
    }
    bf16x8 fa[FM], fb[2][FN];
    auto read_a = [&](int kt, auto ksc, auto halfc) {
        constexpr int ks = decltype(ksc)::value, half = decltype(halfc)::value;
        const unsigned char* st = fw_smem + (kt & 1) * STAGE_BYTES;
#pragma unroll
        for (int i = half * FM / 2; i < (half + 1) * FM / 2; ++i) fa[i] = *(const bf16x8*)(st + offa[ks] + i * 16 * 128);
    };
    auto read_b = [&](int kt, auto ksc, auto halfc) {
        constexpr int ks = decltype(ksc)::value, half = decltype(halfc)::value;
        const unsigned char* st = fw_smem + (kt & 1) * STAGE_BYTES;
#pragma unroll
        for (int j = half * FNH; j < (half ? FN : FNH); ++j) fb[ks][j] = *(const bf16x8*)(st + offb[ks] + j * 16 * 128);
    };
    auto mult = [&](auto ksc, auto halfc) {
        constexpr int ks = decltype(ksc)::value, half = decltype(halfc)::value;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int i = half * FM / 2; i < (half + 1) * FM / 2; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[ks][j], fa[i], acc[i][j], 0, 0, 0);
    };
    // The tail's features of this wave: the 16 from 16 * part on.  TAIL == 1 (a column has at least FN tiles): every tile takes a part of each
    // of its halves, and the two waves of a half take a half of every k-tile each.  TAIL == 2 (at least FN / 2): a wave takes a part
    // and all of k.  Tiles past the last part multiply it once more and store nothing.
    constexpr int TK = TAIL == 2 ? 2 : 1;
    const int my_part = TAIL == 2 ? 2 * tile_row + wm : tile_row, part = min(my_part, FN - 1);
    unsigned offt = 0, offp = 0;
    u32x4 ta[TK];
    bf16x8 tb[TK];
    f32x4 tails[TK];
#pragma unroll
    for (int ks = 0; ks < TK; ++ks) tails[ks] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (TAIL != 0) {
        offt = (unsigned)(((size_t)(M + min(frow, over - 1)) * lda + h * 8) * 2 + (TAIL == 1 ? wm * 64 : 0));
        offp = (TAIL == 1 && wm ? offb[1] : offb[0]) + part * 16 * 128;
    }
    auto ask_tail = [&](int kt) {
        kt = min(kt, nk - 1);
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
        for (int ks = 0; ks < TK; ++ks) ta[ks] = __builtin_amdgcn_raw_buffer_load_b128(ra, offt + ks * 64, kt * 128, 0);
#endif
    };
    auto read_tail = [&](int kt) {
        const unsigned char* st = fw_smem + (kt & 1) * STAGE_BYTES;
#pragma unroll
        for (int ks = 0; ks < TK; ++ks) tb[ks] = *(const bf16x8*)(st + (offp ^ (ks * 64)));     // (the other half of k: its chunk's bit 2 the other way)
    };
    // (The tile's sums fill the accumulation registers; left to the compiler the tail's would push some of them out and in again in every
    // k-tile, with waits for their MFMAs: 57344 x 8192 gated at 2064 rows 1446 us against 1400.  Written out they stay in ordinary registers.  The
    // waits that the compiler sees to for its own MFMAs are owed here: a vector instruction's write of a source, the zeroing of the sums
    // for one, lies two wait states before the MFMA, which stand in front of it; and what reads a result does so seven or more after its MFMA,
    // which the next k-tile's is, and `settle_tail` sees to at the end.)
    auto mult_tail = [&]() {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
        for (int ks = 0; ks < TK; ++ks) asm("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(tails[ks]) : "v"(tb[ks]), "v"(ta[ks]));
#endif
    };
    auto settle_tail = [&]() {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
        for (int ks = 0; ks < TK; ++ks) asm volatile("s_nop 7" : "+v"(tails[ks]));
#endif
    };
    // The order within a step.  A SIMD has this one wave only, so whatever keeps it from issuing its next MFMA leaves the matrix
    // cores idle: loads asked for back to back wait for each other and the other waves' at the address unit (16 cycles
    // each, 16 of them between the four waves), and an MFMA takes 16.  So LDS reads go out in pairs, and every LDS write
    // and every load from memory by itself, with MFMAs after each.  A step's reads are half of the tokens' operands and half of the
    // features', the same number in every step: with all of the tokens' in one step of two LDS is asked for more than it gives in that step.  (57344 x
    // 8192: other numbers of MFMAs after a read, a write and a load within 2 %; reads singly or in fours 1-3 % slower.)
    auto order = [](auto qc, auto readsc, auto multsc) {
        constexpr int q = decltype(qc)::value, LOADS = quarter_of(A_GROUPS, q) + quarter_of(W_GROUPS, q), READS = decltype(readsc)::value, MULTS = decltype(multsc)::value;
        constexpr int after = MULTS >= READS + 3 * LOADS ? 2 : 1;
        static_for<0, READS / 2>([](auto) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, after, 0);
        });
        if constexpr (TAIL != 0 && q == 2) static_for<0, TK>([](auto) {
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        });
        static_for<0, LOADS>([](auto) {
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        });
        __builtin_amdgcn_sched_group_barrier(0x008, MULTS, 0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    // One step (a quarter of a k-tile: half of its k times half of the wave's tokens).  While k-tile kt is multiplied, k-tile kt + 1 goes
    // from registers into the other LDS buffer and k-tile kt + 2 is asked for into the registers that frees.  A quarter written now was
    // asked for a k-tile ago; loads complete in order, so it is there when all but the three other quarters, asked for
    // since, have completed.
    auto step = [&](int kt, auto qc, auto multiply) {
        constexpr int q = decltype(qc)::value;
        using KS = std::integral_constant<int, q / 2>;
        using Odd = std::integral_constant<int, q % 2>;
        if constexpr (q % 2 == 0) read_a(kt, KS{}, I0{});
        read_b(kt, KS{}, Odd{});
        if constexpr (q % 2 == 1) read_a(kt, KS{}, I1{});
        if constexpr (TAIL != 0 && q == 1) read_tail(kt);
        if constexpr (TAIL != 0 && q == 2) { mult_tail(); ask_tail(kt + 1); }
        constexpr int others = A_GROUPS + W_GROUPS - quarter_of(A_GROUPS, q) - quarter_of(W_GROUPS, q);
        wait_vmcnt<others>();
        put(kt + 1, qc);
        ask(kt + 2, qc);
        if constexpr (decltype(multiply)::value) {
            using MK = std::integral_constant<int, q == 0 ? 1 : (q - 1) / 2>;
            mult(MK{}, std::integral_constant<int, 1 - q % 2>{});
        }
        order(qc, std::integral_constant<int, FM / 2 + (q & 1 ? FN - FNH : FNH) + (TAIL != 0 && q == 1 ? TK : 0)>{},
              std::integral_constant<int, FM / 2 * FN>{});
        __builtin_amdgcn_sched_barrier(0);
    };
    // k-tile 0 into LDS, k-tile 1 into registers
    ask(0, I0{}); ask(0, I1{}); ask(0, I2{}); ask(0, I3{});
    wait_vmcnt<0>();
    put(0, I0{}); put(0, I1{}); put(0, I2{}); put(0, I3{});
    ask(1, I0{}); ask(1, I1{}); ask(1, I2{}); ask(1, I3{});
    if constexpr (TAIL != 0) ask_tail(0);
    __syncthreads();               // (waits for the loads of k-tile 1 as well: once)
    // A step multiplies the operands that the steps before it read, and the second half of the features' that it reads itself; the last step's products of a k-tile run in the
    // first step of the next, on operands read before the barrier: the matrix cores work across it.
    auto k_tile = [&](int kt, auto not_first) {
        step(kt, I0{}, not_first);
        step(kt, I1{}, std::true_type{});
        step(kt, I2{}, std::true_type{});
        step(kt, I3{}, std::true_type{});
        block_sync_lds();          // this wave's LDS reads and writes are done, and everybody's
        __builtin_amdgcn_sched_barrier(0);
    };
    k_tile(0, std::false_type{});
    for (int kt = 1; kt < nk; ++kt) k_tile(kt, std::true_type{});
    mult(I1{}, I1{});
    wait_vmcnt<0>();
    __syncthreads();
    band_epilogue<BM, BN, EPI>(acc, fw_smem, out, ldc, M, N, m0, n0, epi);
    if constexpr (TAIL != 0) {
        settle_tail();
        f32x4 tail = tails[0];
        if constexpr (TAIL == 2) tail += tails[TK - 1];
        if constexpr (TAIL == 1) {             // the halves of k together, through LDS behind what the bands used
            f32x4* halves = (f32x4*)(fw_smem + STAGE_BYTES) + wn * 64 + lane;
            if (wm == 1) *halves = tail;
            __syncthreads();
            if (wm == 0) tail += *halves;
        }
        if (my_part < FN && (TAIL == 2 || wm == 0) && frow < over)
            tail_epilogue<EPI>(tail, out, ldc, N, M + frow, n0 + wn * TN + part * 16 + h * 4, epi);
    }
}

// Tiles of 256 x 128 and 128 x 128 whose four multiplying waves have four more beside them, one to a SIMD, that do nothing but bring the operands
// straight into LDS (three k-tiles' places of 48 KB, four of 32).  A wave that multiplies then issues LDS reads and MFMAs alone, its registers hold no operands
// on their way, and half of LDS's work at a k-tile, the writes from registers, goes: 64 MFMAs of a 256 x 128 k-tile take 1024 cycles of a
// SIMD, its reads 768 of LDS and the loads into it 384.  Past the last k-tile the loading waves bring the old values
// that the sums are added to.  Same layout in LDS and same order of k as the kernel above: bitwise the same results.
// What bounds it: the clock under power for long rows (1.15-1.2 PFLOP/s), for short ones the way in and out.  256 x 128 tiles, waves bringing their own -> these, us: 2048 rows
// 4096 x 4096 added to 64.7 -> 57.0 (61.0 without the old values ahead), 4096 x 14336 209.5 -> 202, 2032 rows 3072 x 2048 31.5 -> 28.0, 777 rows 6144 x 4096 49.6 -> 43.3.  128 x 128,
// one block of these to a unit against two of four waves there: 2032 rows 2048 x 2048 added to 36.9 -> 22.7, 2048 x 8192 104 -> 60.
// (The order of reads and MFMAs, two and two, by ones, two and four or reads first, and a raised priority of the multiplying waves: all within 2 %.)
constexpr int fed_stages(int bm) { return bm == 256 ? 3 : 4; }
// The += epilogue with the old values in LDS: piece (band i, wave w, p) is 1 KB, 64 lanes of 16 bytes, number (4 i + w) * 4 + p.  As many bands' as
// two k-tiles' places hold (all of 128 rows, six of eight of 256) lie in `first` and `second`, the others' are read from memory.
template <int BM>
__device__ __forceinline__ void fed_add_epilogue(f32x4 (&acc)[BM / 32][4], unsigned char* mine, const unsigned char* first, const unsigned char* second,
                                                 float* __restrict__ o, int ldc, int M, int N, int m_first, int n_first) {
    constexpr int FM = BM / 32, PER = 4, IN_STAGE = (BM + 128) * 128 / 1024, IN_LDS = 2 * IN_STAGE / 16 < FM ? 2 * IN_STAGE / 16 : FM;      // IN_LDS: bands
    constexpr int ROW_BYTES = 64 * 4 + 16;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), token = lane & 15, g = lane >> 4;
    auto write = [&](auto ic) {
        static_for<0, 4>([&](auto jc) { *(f32x4*)(mine + token * ROW_BYTES + (decltype(jc)::value * 16 + g * 4) * 4) = acc[decltype(ic)::value][decltype(jc)::value]; });
    };
    const int n = n_first + (lane & 15) * 4;
    f32x4 late[FM > IN_LDS ? FM - IN_LDS : 1][PER];          // old values that are still to come
    static_for<IN_LDS, FM>([&](auto ic) {
#pragma unroll
        for (int p = 0; p < PER; ++p) late[decltype(ic)::value - IN_LDS][p] = *(const f32x4*)(o + (size_t)min(m_first + decltype(ic)::value * 16 + p * 4 + g, M - 1) * ldc + min(n, N - 4));
    });
    write(std::integral_constant<int, 0>{});
    static_for<0, FM>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        f32x4 v[PER], old[PER];
        asm volatile("" ::: "memory");
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            v[p] = *(const f32x4*)(mine + (p * 4 + g) * ROW_BYTES + (lane & 15) * 16);
            if constexpr (i < IN_LDS) {
                const int piece = (i * 4 + wave) * 4 + p;
                old[p] = *(const f32x4*)((piece < IN_STAGE ? first + piece * 1024 : second + (piece - IN_STAGE) * 1024) + lane * 16);
            } else old[p] = late[i - IN_LDS][p];
        }
        asm volatile("" ::: "memory");
        if constexpr (i + 1 < FM) write(std::integral_constant<int, i + 1>{});
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            const int m = m_first + i * 16 + p * 4 + g;
            if (m < M && n < N) *(f32x4*)(o + (size_t)m * ldc + n) = old[p] + v[p];
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}
// The q/k/v epilogue of those tiles: the rotation and the cache writes, which were a kernel of their own behind the product (2047 rows, 32 heads on 8 of 64,
// k 2048: 43.3 us for the two, 33.0 in one; 8 of 128 and k 4096 at 1023 rows 66.5 and 55; the product alone 30 and 51).  The rows of q and k
// are also rounded once instead of twice: error against 64 bits 2.34e-3 -> 1.66e-3 of their norm.
struct NothingMore {};
template <int EPI>
using MoreOf = std::conditional_t<EPI == LLMRS_EPI_QKV, QkvEpilogue, NothingMore>;

// The sine and cosine of x, |x| below 2^24: whole turns are taken off by fused multiply-adds with 2 pi in three parts (Cody and Waite's reduction), what
// is left, within half a turn, goes to the vector unit's own instructions, which take turns.
__device__ __forceinline__ void sine_cosine(float x, float& sine, float& cosine) {
    const float n = rintf(x * 0.159154943f);
    float r = __builtin_fmaf(n, -6.28318548f, x);
    r = __builtin_fmaf(n, 1.74845553e-07f, r);
    r = __builtin_fmaf(n, 6.86049956e-15f, r) * 0.159154943f;
    sine = __builtin_amdgcn_sinf(r);
    cosine = __builtin_amdgcn_cosf(r);
}
// What a lane of a multiplying wave asks for before its products: its tokens' positions (fragment i holds token lane % 16 of 16) and the slots of the
// rows of q and k that it stores pieces of (row p * 8 + lane / 8 of a band of 32); below 0 where nothing is to be written.
__device__ __forceinline__ int slot_of_row(const QkvEpilogue& qe, int M, int m) {
    const int slot = qe.write_kv && m < M ? qe.slot_map[m] : -1;
    return slot < qe.num_pages * 16 ? slot : -1;
}
template <int BM>
struct QkvRows {
    static constexpr int FM = BM / 32, BANDS = FM / 2;
    float place[FM];
    int slot[BANDS][4];
};
template <int BM>
__device__ __forceinline__ QkvRows<BM> qkv_rows(const QkvEpilogue& qe, int M, int m_first) {
    const int lane = threadIdx.x & 63;
    QkvRows<BM> rows;
#pragma unroll
    for (int i = 0; i < rows.FM; ++i) rows.place[i] = (float)qe.positions[min(m_first + i * 16 + (lane & 15), M - 1)];
#pragma unroll
    for (int b = 0; b < rows.BANDS; ++b)
#pragma unroll
        for (int p = 0; p < 4; ++p) rows.slot[b][p] = slot_of_row(qe, M, m_first + b * 32 + p * 8 + (lane >> 3));
    return rows;
}
// A wave's 64 features: pairs turn where they lie, in 32-bit, before their one rounding; the rows go through LDS, `mine` (BM / 2 rows, 16 bytes further
// apart than they are long), and those of q and k leave 16 bytes a lane, to the output and to the pages' rows.  Pages of 16 slots, heads
// of a multiple of 8 features.
constexpr int QKV_ROW_BYTES = 64 * 2 + 16;
template <int BM>
__device__ __forceinline__ void qkv_epilogue(f32x4 (&acc)[BM / 32][4], unsigned char* mine, bf16* __restrict__ out, int ldc, int M,
                                             int m_first, int n_first, const QkvEpilogue& qe, const QkvRows<BM>& rows) {
    constexpr int FN = 4;
    const int lane = threadIdx.x & 63, token = lane & 15, four = (lane >> 4) * 4, hd = qe.head_dim;
    const int keys_from = qe.n_heads * hd, values_from = keys_from + qe.n_kv_heads * hd;
    float freq[FN][2];
    unsigned turning = 0;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int n = n_first + j * 16 + four, d = n % hd;
        const bool turns = n < values_from && d < qe.rotary_dim;
        turning |= turns ? 1u << j : 0u;
#pragma unroll
        for (int r = 0; r < 2; ++r) freq[j][r] = turns ? qe.inv_freq[d / 2 + r] : 0.0f;
    }
    // where this lane's pieces of rows go
    const int n = n_first + (lane & 7) * 8, kvh = (n - keys_from) / hd;
    bf16* const k_at = (bf16*)qe.k_cache + ((size_t)kvh * 16 * hd + (n - keys_from - kvh * hd));
    const size_t page_size = (size_t)qe.n_kv_heads * 16 * hd;                     // of all kv heads
    auto write = [&](auto bandc) {
        static_for<0, 2 * FN>([&](auto jc) {
            constexpr int half = decltype(jc)::value / FN, j = decltype(jc)::value % FN, i = 2 * decltype(bandc)::value + half;
            f32x4 v = acc[i][j];
            if (turning >> j & 1) {
#pragma unroll
                for (int r = 0; r < 4; r += 2) {
                    float sn, cs;
                    sine_cosine(rows.place[i] * freq[j][r / 2], sn, cs);
                    const float a = v[r], b = v[r + 1];
                    v[r] = a * cs - b * sn;
                    v[r + 1] = a * sn + b * cs;
                }
            }
            bf16x4 o4;
#pragma unroll
            for (int r = 0; r < 4; ++r) o4[r] = (bf16)v[r];
            *(bf16x4*)(mine + (i * 16 + token) * QKV_ROW_BYTES + (j * 16 + four) * 2) = o4;
        });
    };
    write(std::integral_constant<int, 0>{});
    static_for<0, QkvRows<BM>::BANDS>([&](auto bc) {
        constexpr int band = decltype(bc)::value;
        bf16x8 v[4];
        asm volatile("" ::: "memory");           // (a wave's LDS accesses are carried out in the order it asks for them)
#pragma unroll
        for (int p = 0; p < 4; ++p) v[p] = *(const bf16x8*)(mine + (band * 32 + p * 8 + (lane >> 3)) * QKV_ROW_BYTES + (lane & 7) * 16);
        asm volatile("" ::: "memory");
        if constexpr (band + 1 < QkvRows<BM>::BANDS) write(std::integral_constant<int, band + 1>{});
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int m = m_first + band * 32 + p * 8 + (lane >> 3), slot = rows.slot[band][p];
            if (n < keys_from) {
                if (m < M) *(bf16x8*)(out + (size_t)m * ldc + n) = v[p];
            } else if (n < values_from && slot >= 0) *(bf16x8*)(k_at + (size_t)(slot >> 4) * page_size + (slot & 15) * hd) = v[p];
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}
// Values, [feature][slot] in a page, two bytes a lane with neighbouring lanes on neighbouring tokens, by all eight waves of a block: those of the
// rows that multiplying wave `wave` % 4 left in LDS, the first half of them or the second.  (By the four waves that hold them alone they are what the whole grid waits
// for: 2047 rows of 32 heads on 8 of 64, k 2048, 37.4 us, without the cache writes 30.1.)
template <int BM>
__device__ __forceinline__ void qkv_values(const unsigned char* tile, int wave, int M, int N, int m0, int n0, const QkvEpilogue& qe) {
    constexpr int ROWS = BM / 2, HALF = ROWS / 2, STEP = 64 / HALF;               // a lane: one row and every STEP-th feature
    const int lane = threadIdx.x & 63, of = wave & 3, row = (wave >> 2) * HALF + lane % HALF, hd = qe.head_dim;
    const int values_from = (qe.n_heads + qe.n_kv_heads) * hd, n_first = n0 + (of & 1) * 64;
    const int slot = slot_of_row(qe, M, m0 + (of >> 1) * ROWS + row), from = max(values_from - n_first, 0) + lane / HALF, end = min(N - n_first, 64);
    if (slot < 0) return;
    const unsigned char* mine = tile + of * (ROWS * QKV_ROW_BYTES) + row * QKV_ROW_BYTES;
    // (heads lie one after the other in a page: [kv head][feature][slot])
    bf16* at = (bf16*)qe.v_cache + (size_t)(slot >> 4) * ((size_t)qe.n_kv_heads * 16 * hd) + (slot & 15);
#pragma unroll 4
    for (int lc = from; lc < end; lc += STEP) at[(size_t)(n_first + lc - values_from) * 16] = *(const bf16*)(mine + lc * 2);
}
template <int BM, int EPI>
__global__ __launch_bounds__(512) void gemm_fed_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W,
                                                       void* __restrict__ out, int ldc, int M, int N, int K, int epi, int old_ahead, MoreOf<EPI> more) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char fed_smem[];
    constexpr int BN = 128, STAGES = fed_stages(BM), STAGE_BYTES = (BM + BN) * 128;
    constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16;
    constexpr int A_GROUPS = BM / 8 / 4, W_GROUPS = BN / 8 / 4, LOADS = A_GROUPS + W_GROUPS;      // 8-row groups of a loading wave
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int tile_row, tile_column;
    tile_of_block(K, tile_row, tile_column);
    const int m0 = tile_row * BM, n0 = tile_column * BN;
    // With gridDim.z > 1 (the epilogue then is STORE_F32, `out` the partial sums [gridDim.z][M][N]) a block takes its share of
    // the k-tiles, a contiguous range; no share is empty (the launcher sees to it).
    int nk = K / 64, k_first = 0;
    if (gridDim.z > 1) {
        const int share = (nk + gridDim.z - 1) / gridDim.z;
        k_first = blockIdx.z * share;
        nk = min(share, nk - k_first);
        out = (float*)out + (size_t)blockIdx.z * M * N;
    }
    if (wave >= 4) {
        const int w = wave - 4, lrow = lane >> 3, lslot = lane & 7;
        unsigned oa[A_GROUPS], ow[W_GROUPS];
#pragma unroll
        for (int i = 0; i < A_GROUPS; ++i) {
            int row = (w * A_GROUPS + i) * 8 + lrow;
            oa[i] = (unsigned)(((size_t)min(m0 + row, M - 1) * lda + ((lslot ^ ((row >> 1) & 7)) * 8)) * 2);
        }
#pragma unroll
        for (int i = 0; i < W_GROUPS; ++i) {
            int row = (w * W_GROUPS + i) * 8 + lrow;
            ow[i] = (unsigned)(((size_t)min(n0 + row, N - 1) * K + ((lslot ^ ((row >> 1) & 7)) * 8)) * 2);
        }
#if defined(__HIP_DEVICE_COMPILE__)
        __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, (int)min((size_t)M * lda * 2, (size_t)0xffffffffu), 0x00020000);
        __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)W, 0, (int)min((size_t)N * K * 2, (size_t)0xffffffffu), 0x00020000);
#endif
        // k-tile kt into its place; past the end the old values that the sums are added to (fed_add_epilogue), two places' worth of them
        auto bring = [&](int kt, int place) {
#if defined(__HIP_DEVICE_COMPILE__)
            if (kt < nk) {
                const unsigned base = __builtin_amdgcn_readfirstlane(place * STAGE_BYTES + w * A_GROUPS * 1024);
                const unsigned wbase = __builtin_amdgcn_readfirstlane(place * STAGE_BYTES + BM * 128 + w * W_GROUPS * 1024);
                const int at = (k_first + kt) * 128;
#pragma unroll
                for (int i = 0; i < A_GROUPS; ++i)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void*)(fed_smem + base + i * 1024), 16, oa[i], at, 0, 0);
#pragma unroll
                for (int i = 0; i < W_GROUPS; ++i)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (__attribute__((address_space(3))) void*)(fed_smem + wbase + i * 1024), 16, ow[i], at, 0, 0);
            } else if (EPI == LLMRS_EPI_ACCUM_F32 && old_ahead && kt < nk + 2) {
                __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(out, 0, (int)min((size_t)M * ldc * 4, (size_t)0xffffffffu), 0x00020000);
#pragma unroll
                for (int i = 0; i < LOADS; ++i) {
                    const int piece = (kt - nk) * (4 * LOADS) + w * LOADS + i, band = piece >> 4, cw = (piece >> 2) & 3, p = piece & 3;      // the band is of compute wave cw
                    const int m = min(m0 + (cw >> 1) * (BM / 2) + band * 16 + p * 4 + (lane >> 4), M - 1), n = min(n0 + (cw & 1) * (BN / 2) + (lane & 15) * 4, N - 4);
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(ro, (__attribute__((address_space(3))) void*)(fed_smem + __builtin_amdgcn_readfirstlane(place * STAGE_BYTES + (w * LOADS + i) * 1024)),
                                                             16, (unsigned)(((size_t)m * ldc + n) * 4), 0, 0, 0);
                }
            }
#endif
        };
#pragma unroll
        for (int kt = 0; kt < STAGES; ++kt) bring(kt, kt);
        const int last = nk + (EPI == LLMRS_EPI_ACCUM_F32 && old_ahead ? 2 : 0);
        if (STAGES <= last) wait_vmcnt<(STAGES - 1) * LOADS>(); else wait_vmcnt<0>();
        block_sync_lds();
        int place = 0;
        for (int kt = 0; kt < nk; ++kt) {
            // k-tile kt + 1 is there when all but what has been started since have landed
            if (kt + 1 < nk) {
                if (kt + STAGES - 1 < last) wait_vmcnt<(STAGES - 2) * LOADS>();
                else if (STAGES > 3 && kt + 2 < last) wait_vmcnt<LOADS>();
                else wait_vmcnt<0>();
            }
            block_sync_lds();                        // and k-tile kt has been read
            bring(kt + STAGES, place);
            place = place == STAGES - 1 ? 0 : place + 1;
        }
        wait_vmcnt<0>();                       // (the bands of the results go through the same LDS)
        block_sync_lds();
        if constexpr (EPI == LLMRS_EPI_QKV)
            if (more.write_kv && n0 + BN > (more.n_heads + more.n_kv_heads) * more.head_dim) {
                block_sync_lds();
                qkv_values<BM>(fed_smem, wave, M, N, m0, n0, more);
            }
        return;
    }
    const int wm = wave / 2, wn = wave % 2;
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int frow = lane & 15, h = lane >> 4, sw = (frow >> 1) & 7;
    unsigned offa[2], offb[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        unsigned chunk = (unsigned)(((ks * 4 + h) ^ sw) * 16);
        offa[ks] = (wm * TM + frow) * 128 + chunk;
        offb[ks] = BM * 128 + (wn * TN + frow) * 128 + chunk;
    }
    bf16x8 fa[FM], fb[2][FN];
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    auto step = [&](const unsigned char* st, auto qc, auto multiply) {
        constexpr int q = decltype(qc)::value, ks = q / 2, odd = q % 2;
#pragma unroll
        for (int j = odd * FN / 2; j < (odd + 1) * FN / 2; ++j) fb[ks][j] = *(const bf16x8*)(st + offb[ks] + j * 16 * 128);
#pragma unroll
        for (int i = odd * FM / 2; i < (odd + 1) * FM / 2; ++i) fa[i] = *(const bf16x8*)(st + offa[ks] + i * 16 * 128);
        if constexpr (decltype(multiply)::value) {
            constexpr int mk = q == 0 ? 1 : (q - 1) / 2, half = 1 - odd;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int i = half * FM / 2; i < (half + 1) * FM / 2; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[mk][j], fa[i], acc[i][j], 0, 0, 0);
        }
        static_for<0, (FM + FN) / 4>([](auto) {
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        });
        __builtin_amdgcn_sched_group_barrier(0x008, FM / 2 * FN, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto k_tile = [&](const unsigned char* st, auto not_first) {
        step(st, I0{}, not_first);
        step(st, I1{}, std::true_type{});
        step(st, I2{}, std::true_type{});
        step(st, I3{}, std::true_type{});
        block_sync_lds();
        __builtin_amdgcn_sched_barrier(0);
    };
    [[maybe_unused]] std::conditional_t<EPI == LLMRS_EPI_QKV, QkvRows<BM>, NothingMore> rows;
    if constexpr (EPI == LLMRS_EPI_QKV) rows = qkv_rows<BM>(more, M, m0 + wm * TM);
    block_sync_lds();                          // k-tile 0 is there
    const unsigned char* st = fed_smem;
    k_tile(st, std::false_type{});
    for (int kt = 1; kt < nk; ++kt) {
        st = st == fed_smem + (STAGES - 1) * STAGE_BYTES ? fed_smem : st + STAGE_BYTES;
        k_tile(st, std::true_type{});
    }
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int i = FM / 2; i < FM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[1][j], fa[i], acc[i][j], 0, 0, 0);
    block_sync_lds();
    if constexpr (EPI == LLMRS_EPI_ACCUM_F32) {
        if (old_ahead) {
            auto place = [&](int kt) { return fed_smem + kt % STAGES * STAGE_BYTES; };
            fed_add_epilogue<BM>(acc, place(nk + 2) + wave * (16 * (TN * 4 + 16)), place(nk), place(nk + 1), (float*)out, ldc, M, N, m0 + wm * TM, n0 + wn * TN);
            return;
        }
    }
    if constexpr (EPI == LLMRS_EPI_QKV) {
        static_assert(4 * TM * QKV_ROW_BYTES <= STAGES * STAGE_BYTES && TN == 64, "the whole tile as 16-bit rows lies in LDS");
        qkv_epilogue<BM>(acc, fed_smem + wave * (TM * QKV_ROW_BYTES), (bf16*)out, ldc, M, m0 + wm * TM, n0 + wn * TN, more, rows);
        if (more.write_kv && n0 + BN > (more.n_heads + more.n_kv_heads) * more.head_dim) {
            block_sync_lds();
            qkv_values<BM>(fed_smem, wave, M, N, m0, n0, more);
        }
    } else band_epilogue<BM, BN, EPI>(acc, fed_smem, out, ldc, M, N, m0, n0, epi);
}

// Whether the four-wave tiles can finish this product: the epilogues it has, 16-bit results as whole 16-byte pieces.
static bool fourwave_takes(int epi, const void* out, int ldc, int N) {
    if (epi == LLMRS_EPI_ACCUM_F32 || epi == LLMRS_EPI_STORE_F32) return true;
    if (epi == LLMRS_EPI_STORE) return ldc % 8 == 0 && ((uintptr_t)out & 15) == 0 && N % 8 == 0;
    if (epi_gated(epi)) return ldc % 8 == 0 && ((uintptr_t)out & 15) == 0 && N % 16 == 0;
    return false;
}
template <int BM, int EPI>
static int launch_fed_epi(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi, int splits = 1, const MoreOf<EPI>& more = {}) {
    constexpr int BN = 128;
    static bool configured = false;
    const size_t bytes = (size_t)fed_stages(BM) * (BM + BN) * 128;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_fed_kernel<BM, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return llmrs_fail("gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        configured = true;
    }
    dim3 grid(ceil_div(N, BN), ceil_div(M, BM), splits);
    if (grid.y > 65535) return llmrs_fail("gemm: M=%d is too large for one launch", M);
    const int old_ahead = EPI == LLMRS_EPI_ACCUM_F32 && splits == 1 && N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)out & 15) == 0 && (size_t)M * ldc * 4 < ((size_t)1 << 32);
    gemm_fed_kernel<BM, EPI><<<grid, 512, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi, old_ahead, more);
    return 0;
}
// (operands under 4 GB each, K % 64 == 0, fourwave_takes(epi, ...): the caller's to check, and that no share of k is empty)
template <int BM>
static int launch_fed(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi, int splits = 1) {
    if (epi >= LLMRS_EPI_GLU_CLAMP) return launch_fed_epi<BM, LLMRS_EPI_GLU_CLAMP>(stream, A, lda, W, out, ldc, M, N, K, epi);
    switch (epi) {
        case LLMRS_EPI_STORE: return launch_fed_epi<BM, LLMRS_EPI_STORE>(stream, A, lda, W, out, ldc, M, N, K, epi);
        case LLMRS_EPI_STORE_F32: return launch_fed_epi<BM, LLMRS_EPI_STORE_F32>(stream, A, lda, W, out, ldc, M, N, K, epi, splits);
        case LLMRS_EPI_ACCUM_F32: return launch_fed_epi<BM, LLMRS_EPI_ACCUM_F32>(stream, A, lda, W, out, ldc, M, N, K, epi);
        case LLMRS_EPI_SWIGLU: return launch_fed_epi<BM, LLMRS_EPI_SWIGLU>(stream, A, lda, W, out, ldc, M, N, K, epi);
        default: return llmrs_fail("gemm: the tiles with waves for the loads have no epilogue %d", epi);
    }
}
// over: rows of A and out beyond the M (whole tiles, at least four) that the tiles take along, up to 16
template <int BM, int BN, int EPI, int TAIL = 0>
static int launch_fourwave_epi(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi, int over = 0) {
    if constexpr (TAIL == 0) {
        if (over > 0 && M >= BM * (BN / 32)) return launch_fourwave_epi<BM, BN, EPI, 1>(stream, A, lda, W, out, ldc, M, N, K, epi, over);
        if constexpr (BN > 128)                     // (four tiles are a part for every wave pair of the narrow ones)
            if (over > 0) return launch_fourwave_epi<BM, BN, EPI, 2>(stream, A, lda, W, out, ldc, M, N, K, epi, over);
    }
    static bool configured = false;
    size_t bytes = (size_t)2 * (BM + BN) * 128;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_fourwave_kernel<BM, BN, EPI, TAIL>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return llmrs_fail("gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        configured = true;
    }
    dim3 grid(ceil_div(N, BN), ceil_div(M, BM));
    if (grid.y > 65535) return llmrs_fail("gemm: M=%d is too large for one launch", M);
    if (over > 0 && (over > 16 || M % BM != 0 || TAIL * (int)grid.y < BN / 32))
        return llmrs_fail("gemm: the four-wave tiles cannot take %d rows beyond M=%d along", over, M);
    gemm_fourwave_kernel<BM, BN, EPI, TAIL><<<grid, 256, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi, over);
    return 0;
}
// (operands under 4 GB each, K % 64 == 0, fourwave_takes(epi, ...): the caller's to check)
template <int BM, int BN>
static int launch_fourwave(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi, int over = 0) {
    constexpr int TAIL = BN == 128 ? 1 : 0;       // (256 x 128 tiles without rows to take along are launch_fed's)
    if (TAIL == 1 && over == 0) return launch_fed<256>(stream, A, lda, W, out, ldc, M, N, K, epi);
    if (epi >= LLMRS_EPI_GLU_CLAMP) return launch_fourwave_epi<BM, BN, LLMRS_EPI_GLU_CLAMP, TAIL>(stream, A, lda, W, out, ldc, M, N, K, epi, over);
    switch (epi) {
        case LLMRS_EPI_STORE: return launch_fourwave_epi<BM, BN, LLMRS_EPI_STORE, TAIL>(stream, A, lda, W, out, ldc, M, N, K, epi, over);
        case LLMRS_EPI_STORE_F32: return launch_fourwave_epi<BM, BN, LLMRS_EPI_STORE_F32, TAIL>(stream, A, lda, W, out, ldc, M, N, K, epi, over);
        case LLMRS_EPI_ACCUM_F32: return launch_fourwave_epi<BM, BN, LLMRS_EPI_ACCUM_F32, TAIL>(stream, A, lda, W, out, ldc, M, N, K, epi, over);
        case LLMRS_EPI_SWIGLU: return launch_fourwave_epi<BM, BN, LLMRS_EPI_SWIGLU, TAIL>(stream, A, lda, W, out, ldc, M, N, K, epi, over);
        default: return llmrs_fail("gemm: the four-wave tiles have no epilogue %d", epi);
    }
}

// Into how many parts the k range is split over blocks (1: not at all), by the product's shape alone.
// 17 to 64 rows (few-row kernel, 64 features per block): when the features give no more than 64
// blocks, until there are 256 of them, each part at least 16 k-blocks long (measured at 64 rows:
// 4096 x 14336 in 4 parts 35 us, in 8 parts 42; 2048 x 8192 in 8 parts 18 us, in 4 parts 23; at 32
// rows 4096 x 14336 40 -> 28 us, 2048 x 8192 24 -> 14; it no longer pays for N = 6144).
static int skinny_splits(int N, int K) {
    int blocks = ceil_div(N, 64), nkb = ceil_div(K, 64), splits = 1;
    while (blocks <= 64 && blocks * splits < 256 && splits < 16 && nkb / (splits * 2) >= 8) splits *= 2;
    return splits;
}
// (128 x 128 tiles for 17 to 64 rows, and for operands of 4 GB and more.)
// Up to 256 rows whose 128 x 128 tiles are no more than the compute units: one block of eight waves per
// unit with four k-tiles in LDS (three on their way) instead of two blocks of four waves with two
// k-tiles each.  A tile's loads into LDS take longer than its MFMAs, and with few blocks per unit
// the deeper pipeline is what keeps them coming (measured, 128 rows at the 8B shapes: qkv 21.9 -> 19.7 us,
// o 21.3 -> 18.6, gate/up 76.6 -> 64.8, down 43.7 -> 36.6; 256 rows: o 25.8 -> 21.9, down 56.4 -> 50.9;
// with more tiles than units, or more rows, the two blocks win).
static bool deep_tiles(int M, int N, int K) {
    return K % 64 == 0 && M <= 256 && (long)ceil_div(M, 128) * ceil_div(N, 128) <= llmrs_compute_units();
}
// Above (128 x 128 tiles): until the tiles fill the places (two to a compute unit, or one where the
// deep pipeline runs), each part at least 8 k-tiles long.
static int tiled_splits(int M, int N, int K) {
    if (K % 64) return 1;
    long tiles = (long)ceil_div(M, 128) * ceil_div(N, 128);
    long places = (long)llmrs_compute_units() * (deep_tiles(M, N, K) ? 1 : 2);
    int nk = K / 64, splits = 1;
    while (tiles * splits * 2 <= places && splits < 16 && nk / (splits * 2) >= 8) splits *= 2;
    return splits;
}
// The 128 x 128 tiles of a product, in whichever of the two forms its shape asks for.
static int launch_tiles_128(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc,
                            int M, int N, int K, int epi, int splits, float* partial, const NextNorm* next = nullptr,
                            bool finish = true) {
    if (deep_tiles(M, N, K)) return launch_dma<128, 128, 2, 4, 4>(stream, A, lda, W, out, ldc, M, N, K, epi, splits, partial, next, finish);
    return launch_dma<128, 128, 2, 2, 2>(stream, A, lda, W, out, ldc, M, N, K, epi, splits, partial, next, finish);
}
// More than 64 rows, where square large tiles would not fill the device: tiles of 256 x 128 or of 128 x 128 with waves of their own for the loads, a
// block to a unit, with k split over 1 to 16 blocks, whichever takes the least time (us) by what was measured: a part for every k-tile
// of a round, a part that follows how full the device is (the clock follows the power), a block's way in and out, the operands' first trip from
// memory, and for a split product the kernel that adds the parts up, or the norm's own kernel where a product that adds to the stream is not split.
// (603 products of 65 to 4200 rows, 160 to 28,000 features and k of 64 to 14336, every epilogue, weights from memory: the plans chosen take 1.010 of the
// best of all nine, and 0.8 of the time of the 128 x 128 and 256 x 128 tiles before, whose waves brought their own operands; those were the
// faster ones nowhere from 512 rows on.  us, before and now: 2032 rows 2048 x 2048 added to, with the norm 39.0 -> 33.1, 2048 x 8192 87.6 -> 75.5,
// 3072 x 2048 33.0 -> 29.4; 1024 rows 4096 x 4096 with the norm 51.1 -> 48.2, 900 rows 3072 x 2048 28.5 -> 18.0, 450 rows 6144 x 4096 46.9 -> 33.9, 200 rows 4096 x 14336
// 48.5 -> 43.7, 96 rows 2048 x 2048 16.0 -> 13.9.  The worst choice: 1047 rows 4096 x 10368, 157 and 113 in two parts.)
// The two operands' sizes, under 4 GB, are looked at where it is launched.
struct MidTiles {
    int rows;          // of a tile: 256 or 128
    int splits;
    double time;
};
static MidTiles mid_tiles(int M, int N, int K, int epi, bool may_split = true) {
    const int cus = llmrs_compute_units(), nk = K / 64;
    MidTiles best{128, 1, 1e30};
    if (K % 64) return best;
    const double mn = (double)M * N * 1e-6, mk = (double)M * K * 2e-6, nkb = (double)N * K * 2e-6;
    const bool adds = epi == LLMRS_EPI_ACCUM_F32;
    for (int rows = 256; rows >= 128; rows /= 2)
        for (int z = 1; z == 1 || (may_split && z <= 16 && nk / z >= 8); z *= 2) {
            const int share = ceil_div(nk, z);
            if ((z - 1) * share >= nk) continue;                      // (no share may be empty)
            const long blocks = (long)ceil_div(M, rows) * ceil_div(N, 128) * z;
            const double rounds = (double)ceil_div(blocks, (long)cus), full = (double)blocks / cus;
            const bool stores_f32 = epi == LLMRS_EPI_STORE_F32 || z > 1;
            double t = rows == 256 ? rounds * (3.2 + 0.42 * share + (stores_f32 ? 1.9 : adds ? 3.2 : 0.0)) + 0.28 * share * full + 0.16 * mk + 0.06 * nkb
                                   : rounds * (2.3 + 0.28 * share + (stores_f32 ? 1.0 : adds ? 1.9 : 0.0)) + 0.18 * share * full + 0.05 * mk + 0.085 * nkb;
            t += 3.0;
            if (z > 1) t = 1.06 * (t + 2.5 + 0.2 * mn * (4 * z + (adds ? 8 : epi == LLMRS_EPI_STORE_F32 ? 4 : epi_gated(epi) ? 1 : 2)));
            else if (adds) t += 2.0 + 1.33 * mn;
            if (t < best.time) best = MidTiles{rows, z, t};
        }
    return best;
}
static int launch_mid(hipStream_t stream, int rows, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi, int splits = 1) {
    return rows == 256 ? launch_fed<256>(stream, A, lda, W, out, ldc, M, N, K, epi, splits) : launch_fed<128>(stream, A, lda, W, out, ldc, M, N, K, epi, splits);
}
// As parts of its sum, for whatever epilogue follows: the most that any of them asks for (so much room is what a caller brings).
static int most_splits(int M, int N, int K) {
    int most = 1;
    for (int epi : {LLMRS_EPI_STORE, LLMRS_EPI_STORE_F32, LLMRS_EPI_ACCUM_F32, LLMRS_EPI_SWIGLU}) most = std::max(most, mid_tiles(M, N, K, epi).splits);
    return most;
}
// 17..64 rows on a weight of middling width (more than 4096 features, fewer than the wide ones that
// get blocks of many feature tiles): the 128 x 128 tiles with k split over blocks.  Where they add to the stream their finish also
// does the norm that follows; their tokens' rows are read less often than the ring's blocks of 32 features read them, which pays at
// long rows and many tokens (ring against tiles, us: 8192 x 28672 111 / 90 at 20 rows, 133 / 99 at 64; 10240 x 8192 60 / 52 at 64,
// 12288 x 4096 35.6 / 34.3 at 64).
static bool few_rows_take_tiles(int M, int N, int K) {
    return M > 16 && M <= 64 && N > 4096 && N < 16384 && K % 64 == 0 && tiled_splits(M, N, K) > 1;
}
// Of those the products with short rows that store their results or gate them are better off with the ring (tiles with their finish -> ring, us:
// 17 rows 8192 x 2048 15.3 -> 11.3, 10240 x 4096 27.8 -> 22.0; over 4608 to 16000 features a ratio of 0.67 at K = 1024 whatever
// the rows, 0.76-0.98 at 2048 to 4096 and up to 32 rows; with more rows or longer ones some gain and some lose up to 22 %).
// 33 to 48 rows read theirs often enough for the tiles to win over many features with rows of 2048 to 4096 (ring / tiles, 48 rows 14336 x 2560
// 1.12, 13824 x 3584 1.09, 9216 x 2560 1.05; 40 rows 14336 x 2560 1.04, 12288 x 2560 0.98; at K = 2048 0.92-0.98, at 4096 0.80-1.0).
static bool ring_stores_faster(int M, int N, int K) {
    const bool tiles_between = M > 32 && N > (M <= 40 ? 12288 : 8192) && K > 2048 && K < 4096;
    return K <= (M <= 48 ? 4096 : 1024) && !tiles_between;
}
// Whether a product of more than 64 rows goes to the tiles of `mid_tiles` (the launcher asks the same).
static bool mid_takes(int M, int N, int K) { return M > 64 && K % 64 == 0 && (long)ceil_div(M, 256) * ceil_div(N, 256) < 160; }
// What `mid_tiles` says of a product that goes there: 100 times the splits and 1 or 2 for tiles of 128 or 256 rows; 0 where it does not go.
extern "C" int llmrs_gemm_mid_plan(int M, int N, int K, int epi) {
    if (!mid_takes(M, N, K)) return 0;
    const MidTiles plan = mid_tiles(M, N, K, epi);
    return 100 * plan.splits + plan.rows / 128;
}
// Room (in floats) for the partial sums of a product that would be split: what the caller should bring.  (A little of it
// where none is split but the norm that follows can be finished, which is asked for by bringing some.)
extern "C" long llmrs_gemm_workspace_floats(int M, int N, int K) {
    if (M > 16 && M <= 64) {
        int s = few_rows_take_tiles(M, N, K) ? tiled_splits(M, N, K) : skinny_splits(N, K);
        return s > 1 ? (long)s * M * N : 0;
    }
    if (M >= 1024 && M % 256 > 16 && M % 256 <= 64 && K % 64 == 0 && (long)(M / 256) * ceil_div(N, 256) >= 160) {
        int s = skinny_splits(N, K);            // the rows beyond whole large tiles go to the kernel for few rows
        return s > 1 ? (long)s * (M % 256) * N : 0;
    }
    if (M > 64 && (long)ceil_div(M, 256) * ceil_div(N, 256) < 160) {
        int s = most_splits(M, N, K);
        long own = s > 1 ? (long)s * M * N : mid_takes(M, N, K) ? 64 : 0;
        // a few rows beyond whole 128-row tiles may go to the kernel for few rows, and the whole tiles be split then
        int over128 = M % 128;
        if (M >= 1024 && over128 > 0 && over128 <= 64 && K % 64 == 0)
            own = std::max(own, std::max(llmrs_gemm_workspace_floats(M - over128, N, K), llmrs_gemm_workspace_floats(over128, N, K)));
        return own;
    }
    return 0;
}

// 17 rows or more whose sums are split over blocks: the kernel that adds the parts up can finish the following norm.  So can, in a launch
// behind the product, every product of more than 64 rows that goes to the tiles of `mid_tiles`, split or not.
extern "C" int llmrs_gemm_norms_whole(int M, int N, int K) {
    if (!(M > 16 && N >= 4 && N % 4 == 0 && N <= 16384 && K % 8 == 0)) return 0;
    return M <= 64 ? llmrs_gemm_workspace_floats(M, N, K) > 0 : mid_takes(M, N, K);
}

// The product as parts of its sum over k, [parts][M][N] 32-bit in `workspace`, for a caller that adds them up itself
// (the rotation and cache write after the q/k/v product does, and saves the kernel that would): only where this
// file would split such a product over blocks anyway.  Returns the number of parts, 0 when the product is not
// one of those (nothing was launched), -1 on error.
int llmrs_gemm_bf16_split_parts(hipStream_t stream, const bf16* A, int lda, const bf16* W, int M, int N, int K,
                                void* workspace, size_t workspace_bytes) {
    if (K % 64 || lda % 8 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15) || workspace == nullptr || M > 512) return 0;
    const bool small = (size_t)M * lda * 2 < ((size_t)1 << 32) && (size_t)N * K * 2 < ((size_t)1 << 32);
    if (M > 64 ? (long)ceil_div(M, 256) * ceil_div(N, 256) >= 160 || !small : !few_rows_take_tiles(M, N, K)) return 0;
    const MidTiles plan = M > 64 ? mid_tiles(M, N, K, LLMRS_EPI_STORE) : MidTiles{0, tiled_splits(M, N, K), 0.0};
    const int splits = plan.splits;
    if (splits <= 1 || workspace_bytes < (size_t)splits * M * N * sizeof(float)) return 0;
    const int rc = plan.rows != 0 ? launch_mid(stream, plan.rows, A, lda, W, workspace, N, M, N, K, LLMRS_EPI_STORE_F32, splits)
                                  : launch_tiles_128(stream, A, lda, W, nullptr, N, M, N, K, LLMRS_EPI_STORE, splits, (float*)workspace, nullptr, false);
    if (rc != 0) return -1;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { llmrs_fail("gemm (mfma): launch failed: %s", hipGetErrorString(e)); return -1; }
    return splits;
}

// More than 64 rows of a q/k/v product whose rotation and cache write its tiles do themselves: those of `mid_tiles` that are not
// split (there the rotation adds the parts up as it reads them).  The four-wave tiles of 256 features that take more rows keep the kernel behind them: with
// this epilogue they were no faster, 106 us either way at 2048 x 6144 x 4096.  1, 0 where the product goes another way, -1 on error.
static int qkv_in_tiles(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, const QkvEpilogue& qkv) {
    const bool small = (size_t)M * lda * 2 < ((size_t)1 << 32) && (size_t)N * K * 2 < ((size_t)1 << 32);
    if (!mid_takes(M, N, K) || !small || qkv.page_size != 16 || qkv.head_dim % 8 || ldc % 8 || (((uintptr_t)out | (uintptr_t)qkv.k_cache) & 15)) return 0;
    const int over = M % 128;
    const MidTiles plan = mid_tiles(M, N, K, LLMRS_EPI_STORE);
    // (the rows beyond whole tiles that the launcher below gives to the kernel for few rows go there)
    if (plan.splits > 1 || (M >= 1024 && over > 0 && over <= 64 && plan.time - mid_tiles(M - over, N, K, LLMRS_EPI_STORE).time >= 30.0)) return 0;
    const int rc = plan.rows == 256 ? launch_fed_epi<256, LLMRS_EPI_QKV>(stream, A, lda, W, out, ldc, M, N, K, LLMRS_EPI_QKV, 1, qkv)
                                    : launch_fed_epi<128, LLMRS_EPI_QKV>(stream, A, lda, W, out, ldc, M, N, K, LLMRS_EPI_QKV, 1, qkv);
    if (rc != 0) return -1;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { llmrs_fail("gemm (mfma): launch failed: %s", hipGetErrorString(e)); return -1; }
    return 1;
}

int llmrs_gemm_bf16_mfma(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc,
                         int M, int N, int K, int epi, void* workspace, size_t workspace_bytes,
                         const QkvEpilogue* qkv, const RowScale* scale, const NextNorm* next) {
    if (K % 8 || lda % 8 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15)) {
        if (scale != nullptr || next != nullptr) { llmrs_fail("gemm: a deferred norm needs rows of a multiple of 8 values, 16-byte aligned"); return -1; }
        return 0;
    }
    const bool whole = next != nullptr && next->eps > 0.0f;      // the norm that follows is finished by the kernel that adds the parts up
    if (whole) {
        bool ok = scale == nullptr && epi == LLMRS_EPI_ACCUM_F32 && llmrs_gemm_norms_whole(M, N, K) && workspace != nullptr &&
                  workspace_bytes >= (size_t)llmrs_gemm_workspace_floats(M, N, K) * sizeof(float) && next->y != nullptr &&
                  next->weight != nullptr && next->ldy >= N && next->ldy % 4 == 0 && ((uintptr_t)next->y & 7) == 0 &&
                  ((uintptr_t)next->weight & 15) == 0 && ldc % 4 == 0 && ((uintptr_t)out & 15) == 0 && ((uintptr_t)workspace & 15) == 0;
        if (!ok) { llmrs_fail("gemm: a norm finished by a split product needs the += epilogue, 17 rows or more of a shape that is split, its workspace and aligned rows, got M=%d N=%d K=%d epilogue %d", M, N, K, epi); return -1; }
    } else if ((scale != nullptr || next != nullptr) && !llmrs_gemm_defers_norm(M, N, K)) {
        llmrs_fail("gemm: a deferred norm is taken for up to 16 rows, got M=%d N=%d K=%d epilogue %d", M, N, K, epi);
        return -1;
    }
    if (epi == LLMRS_EPI_QKV) {   // four features of a head at a time: aligned rows
        if (qkv == nullptr || !llmrs_qkv_by_fours(qkv->head_dim, qkv->rotary_dim) || ldc % 4 || ((uintptr_t)out & 7) ||
            ((uintptr_t)qkv->k_cache & 7))
            return 0;
        if (M > 64) return scale != nullptr ? 0 : qkv_in_tiles(stream, A, lda, W, out, ldc, M, N, K, *qkv);
        // long rows and many tokens: the tiles with k split over blocks are so much faster that
        // the separate rotation kernel is paid for (10240 x 8192 at 64 rows: 60 us in the ring, 52 + 6; the tiles' parts are added by the rotation)
        // (with rows of 4096 the same route gains nothing: a decode step of the 8B shape at 64 requests 7.60 -> 7.55 ms,
        // at 40 and 48 requests none or a loss)
        if (M > 32 && K >= 8192 && few_rows_take_tiles(M, N, K)) return 0;
    }
    int rc = 0;
    if (M <= 16) {
        int took = llmrs_gemm_few_bf16(stream, A, lda, W, out, ldc, M, N, K, epi, qkv, scale, next);
        if (took <= 0) return took;
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) { llmrs_fail("gemm (mfma): launch failed: %s", hipGetErrorString(e)); return -1; }
        return 1;
    }
    bool tiles_for_few = false;
    if (epi != LLMRS_EPI_QKV && few_rows_take_tiles(M, N, K) && (epi == LLMRS_EPI_ACCUM_F32 || !ring_stores_faster(M, N, K))) {
        int splits = tiled_splits(M, N, K);
        tiles_for_few = workspace != nullptr && workspace_bytes >= (size_t)splits * M * N * sizeof(float);
    }
    if (tiles_for_few) {
        rc = launch_tiles_128(stream, A, lda, W, out, ldc, M, N, K, epi, tiled_splits(M, N, K), (float*)workspace, next);
    } else if (M <= 64) {
        // Features per block grow with N: a block reads its tokens' rows again, which costs once M is large, but a weight
        // with few rows needs small blocks to have enough of them; the narrowest ones have their k-blocks shared out over blocks
        // as well.  (Measured on MI355X at the 1B and 8B shapes.)
        const bool wide = N >= 16384;
        const int cus = llmrs_compute_units(), splits = skinny_splits(N, K);
        const bool split = splits > 1 && epi != LLMRS_EPI_QKV && workspace != nullptr && workspace_bytes >= (size_t)splits * M * N * sizeof(float);
        if (whole && splits <= 1) { llmrs_fail("gemm: M=%d N=%d K=%d is not split after all: the norm cannot be finished here", M, N, K); return -1; }
        // A wide weight's blocks take 7 or 4 feature tiles: whichever number of blocks fills the
        // device's compute units more evenly (28672 features are 256 blocks of 7 tiles).
        auto evenness = [&](int nt) { int b = ceil_div(N, 16 * nt); return (double)b / ((double)ceil_div(b, cus) * cus); };
        auto rows_of = [&](auto tiles) {
            constexpr int MT = decltype(tiles)::value;
            // (and, adding to the stream, the shortest rows of narrow weights with up to 32 tokens, which come to a few k-blocks a wave and no
            // steady state of the ring: 17 rows 512 x 512 4.0 us, in the ring 4.4, 1024 x 256 3.45 and 3.7; 40 rows are better off there)
            if (K % 64 || (MT == 2 && N <= 4096 && K <= 512 && epi == LLMRS_EPI_ACCUM_F32)) {
                // Eight waves where rows are long, and the more k-blocks on their way the fewer features and tokens a block has; a walk
                // along k that begins at a place of the block's own for wide weights and long rows (17 rows 8192 x 8224: 32.8 us,
                // in step 49.8; 28672 x 4128: 49.8, in step and in blocks of four tiles 61.9; 64 rows 3072 x 96: 3.4, with eight waves 4.0).
                const int rot = wide ? 16 * (evenness(7) >= evenness(4) ? 7 : 4) : (K >= 8192 ? 64 : 0);
                const bool eight = K >= 2048;
#define SKINNY(NT, NW, U, LAST) launch_skinny<MT, NT, NW, U, LAST>(stream, A, lda, W, out, ldc, M, N, K, epi, qkv, 1, nullptr, rot)
                if (split) launch_skinny<MT, 4, 8, 1>(stream, A, lda, W, out, ldc, M, N, K, epi, nullptr, splits, (float*)workspace, 0, next);
                else if (wide) { if (evenness(7) >= evenness(4)) SKINNY(7, 4, 1, 16); else SKINNY(4, 4, 2, 16); }
                else if (N > 4096) {
                    if (eight && llmrs_half_tile_blocks(N, 32, cus)) SKINNY(2, 8, (MT == 2 ? 2 : 1), 8);
                    else if (eight) SKINNY(2, 8, (MT == 2 ? 2 : 1), 16);
                    else SKINNY(2, 4, 2, 16);
                }
                else { if (eight) SKINNY(1, 8, (MT == 2 ? 4 : 2), 16); else SKINNY(1, 4, (MT == 2 ? 4 : 2), 16); }
#undef SKINNY
                return;
            }
#define RING(NT, LAST, KSUB, ROT) launch_ring<MT, NT, LAST, KSUB>(stream, A, lda, W, out, ldc, M, N, K, epi, qkv, 1, nullptr, ROT)
#define RING_SPLIT(NT, KSUB) launch_ring<MT, NT, 16, KSUB>(stream, A, lda, W, out, ldc, M, N, K, epi, nullptr, splits, (float*)workspace, apart, next)
            // (shares of rows of a multiple of 16 KB begin in step: up to 32 rows, whose weights are most of what is read, want them apart.  17 rows 4096 x
            // 16384 38.6 -> 30.1 us, 4096 x 8192 23.1 -> 19.4, 2048 x 16384 0.88 of the time; other rows 0.92-1.04 of it, with 64 rows long ones 1.12.)
            const int apart = MT == 2 && K % 8192 == 0 ? 64 : 0;
            // (64 rows: 2048 x 2048, 128 blocks of 64 features with their shares of k, 12.0 us, 256 of 32 10.4; 2048 x 8192 16.6 and 18.5)
            if (split) { if (ceil_div(N, 64) * splits >= cus) RING_SPLIT(4, 1); else RING_SPLIT(2, 2); }
            else if (wide) { if (evenness(7) >= evenness(4)) RING(7, 16, 1, 112); else RING(4, 16, 1, 64); }
            // 6144 features are 256 blocks of 24 (a tile and a half), 3072 192 of 16
            else if (N > 4096) { if (llmrs_half_tile_blocks(N, 32, cus)) RING(2, 8, 1, 0); else RING(2, 16, 1, 0); }
            else RING(1, 16, 2, 0);
#undef RING
#undef RING_SPLIT
        };
        if (M <= 32) rows_of(std::integral_constant<int, 2>{});
        else if (M <= 48) rows_of(std::integral_constant<int, 3>{});
        else rows_of(std::integral_constant<int, 4>{});
    } else {
        // K % 64 == 0: tiles whose operands are brought into LDS whole k-tiles of 64 ahead.  Other K: through
        // registers, with zero-filled tails.
        // 256 x 256 tiles where they fill most of the device (from 160 of them on; below, the smaller ones take less time, above they
        // take 1.01 to 1.27 of it at 41 of 43 sizes); else 256 x 128 or 128 x 128, with the k range split over blocks when even
        // those are too few (mid_tiles).
        // One large tile runs on a compute unit at a time, so a grid of them works in rounds and the
        // last round may be far from full (896 tiles on 256 units: 3.5 rounds cost 4).  Then the large
        // tiles get the features that make whole rounds and the smaller ones the rest.
        long m_tiles = ceil_div(M, 256), big_tiles = m_tiles * ceil_div(N, 256);
        int cus = llmrs_compute_units();
        // A few rows beyond whole tiles (a prompt portion of 2048 tokens beside 16 decoded ones)
        // would cost another row of tiles in full: they go to the kernel for few rows instead,
        // which reads the weight once more at memory speed.
        int over = M % 256;
        // Up to 16 of them go along with the four-wave tiles, where those take the product (2-4 % of the tiles' time, at 1032 to 8208 rows less
        // than the few-row kernel's 8-14; beyond 256 x 128 tiles of fewer than 160 large ones both come to the same, and the few-row kernel stays).
        // operands under 4 GB are read through buffer descriptors (32-bit offsets), 1-4 % faster
        const bool small = (size_t)M * lda * 2 < ((size_t)1 << 32) && (size_t)N * K * 2 < ((size_t)1 << 32);
        const bool over_beside = K % 64 == 0 && M >= 1024 && over > 0 && over <= 64 && (m_tiles - 1) * ceil_div(N, 256) >= 160;
        int along = 0;
        if (over_beside && over <= 16 && small && fourwave_takes(epi, out, ldc, N)) {
            along = over;
            M -= over;
            m_tiles -= 1;
            big_tiles = m_tiles * ceil_div(N, 256);
        } else if (over_beside) {
            size_t elt = (epi == LLMRS_EPI_STORE_F32 || epi == LLMRS_EPI_ACCUM_F32) ? sizeof(float) : sizeof(bf16);
            int whole_rows = M - over;
            rc = llmrs_gemm_bf16_mfma(stream, A, lda, W, out, ldc, whole_rows, N, K, epi, workspace, workspace_bytes, qkv);
            if (rc != 1) return rc;
            return llmrs_gemm_bf16_mfma(stream, A + (size_t)whole_rows * lda, lda, W, (char*)out + (size_t)whole_rows * ldc * elt,
                                        ldc, over, N, K, epi, workspace, workspace_bytes, qkv);
        }
        // (up to 128 rows a 256-row tile would be half empty; 257-384 rows are still faster on two rows of
        // large tiles than on three of small ones: the lm head at 300 rows 640 against 750 us)
        if (K % 64 == 0 && big_tiles >= 160 && M > 128) {
            // square tiles: four waves with 128 x 128 outputs each where their epilogues and loads allow, else the
            // eight waves in two groups
            const bool four = small && fourwave_takes(epi, out, ldc, N);
            long whole = big_tiles / cus * cus, rest = big_tiles - whole;
            int n_split = (int)(whole / m_tiles) * 256;        // features of the whole rounds
            // (the features beyond whole rounds run on 128 x 128 tiles, two to a unit, a round of which takes about 0.62 of
            // a round of large tiles: when they come to more than one such round, a last round of large tiles that is
            // not full may be the shorter way: the o and down products at 6144 rows, 1.5 rounds of large tiles)
            long small_blocks = (long)ceil_div(N - n_split, 128) * ceil_div(M, 128);
            bool split_pays = (double)(whole / cus) + 0.62 * ceil_div(small_blocks, 2L * cus) < (double)ceil_div(big_tiles, (long)cus);
            if (n_split > 0 && n_split < N && rest > 0 && 2 * rest <= cus + cus / 4 && split_pays) {
                size_t elt = (epi == LLMRS_EPI_STORE_F32 || epi == LLMRS_EPI_ACCUM_F32) ? sizeof(float) : sizeof(bf16);
                void* out_rest = (char*)out + (size_t)(epi_gated(epi) ? n_split / 2 : n_split) * elt;
                rc = four && fourwave_takes(epi, out, ldc, n_split)
                         ? launch_fourwave<256, 256>(stream, A, lda, W, out, ldc, M, n_split, K, epi, along)
                     : small ? launch_pingpong<256, 256, 2, 4, true>(stream, A, lda, W, out, ldc, M, n_split, K, epi)
                             : launch_pingpong<256, 256, 2, 4, false>(stream, A, lda, W, out, ldc, M, n_split, K, epi);
                if (rc == 0) {
                    const bool fed = four && fourwave_takes(epi, out_rest, ldc, N - n_split);
                    if (fed && mid_tiles(M, N - n_split, K, epi, false).rows == 256)
                        rc = launch_fourwave<256, 128>(stream, A, lda, W + (size_t)n_split * K, out_rest, ldc, M, N - n_split, K, epi, along);
                    else {
                        rc = fed ? launch_fed<128>(stream, A, lda, W + (size_t)n_split * K, out_rest, ldc, M, N - n_split, K, epi)
                                 : launch_dma<128, 128, 2, 2, 2>(stream, A, lda, W + (size_t)n_split * K, out_rest, ldc, M, N - n_split, K, epi);
                        if (rc == 0 && along > 0) {
                            int took = llmrs_gemm_bf16_mfma(stream, A + (size_t)M * lda, lda, W + (size_t)n_split * K,
                                                            (char*)out_rest + (size_t)M * ldc * elt, ldc, along, N - n_split, K, epi, nullptr, 0);
                            if (took != 1) return took < 0 ? -1 : (llmrs_fail("gemm: nothing takes the last %d rows of N=%d K=%d", along, N, K), -1);
                        }
                    }
                }
            } else if (long t192 = m_tiles * ceil_div(N, 192); rest > 0 && t192 % cus == 0) {
                // 256 x 192 tiles where they come to whole rounds of the device and the square ones do not: the
                // q/k/v product of the 8B shape at 2048 rows is 192 square tiles on 256 units, or 256 of these
                // (four waves of 128 x 96: 87 us, against 100 for the eight waves of 64 x 96)
                rc = four ? launch_fourwave<256, 192>(stream, A, lda, W, out, ldc, M, N, K, epi, along)
                   : small ? launch_pingpong<256, 192, 4, 2, true>(stream, A, lda, W, out, ldc, M, N, K, epi)
                           : launch_pingpong<256, 192, 4, 2, false>(stream, A, lda, W, out, ldc, M, N, K, epi);
            } else {
                rc = four ? launch_fourwave<256, 256>(stream, A, lda, W, out, ldc, M, N, K, epi, along)
                     : small ? launch_pingpong<256, 256, 2, 4, true>(stream, A, lda, W, out, ldc, M, N, K, epi)
                             : launch_pingpong<256, 256, 2, 4, false>(stream, A, lda, W, out, ldc, M, N, K, epi);
            }
        } else if (K % 64 == 0) {
            // The same for the 128 x 128 tiles, whose blocks run two to a compute unit: a few rows beyond whole
            // tiles that cost them another round of the device, or the split of k that filled it, go to the kernel
            // for few rows (the o and down products of the 8B shape: 2049 rows 526 -> about 350 us, 1025 rows 287 -> 240).
            // By the time of the plans for all rows and for the whole tiles' (us, mid_tiles).
            auto plan_of = [&](int rows) {
                MidTiles plan = mid_tiles(rows, N, K, epi);
                if (plan.splits > 1 && (workspace == nullptr || workspace_bytes < (size_t)plan.splits * rows * N * sizeof(float)))
                    plan = mid_tiles(rows, N, K, epi, false);
                return plan;
            };
            int over128 = M % 128;
            if (M >= 1024 && over128 > 0 && over128 <= 64) {
                if (plan_of(M).time - plan_of(M - over128).time >= 30.0) {
                    size_t elt = (epi == LLMRS_EPI_STORE_F32 || epi == LLMRS_EPI_ACCUM_F32) ? sizeof(float) : sizeof(bf16);
                    int whole_rows = M - over128;
                    rc = llmrs_gemm_bf16_mfma(stream, A, lda, W, out, ldc, whole_rows, N, K, epi, workspace, workspace_bytes, qkv);
                    if (rc != 1) return rc;
                    rc = llmrs_gemm_bf16_mfma(stream, A + (size_t)whole_rows * lda, lda, W, (char*)out + (size_t)whole_rows * ldc * elt,
                                              ldc, over128, N, K, epi, workspace, workspace_bytes, qkv);
                    if (rc == 1 && whole) launch_norm_rows(stream, out, ldc, M, N, *next);
                    return rc;
                }
            }
            const MidTiles plan = plan_of(M);
            const int splits = plan.splits;
            if (small && splits > 1) {
                rc = launch_mid(stream, plan.rows, A, lda, W, workspace, N, M, N, K, LLMRS_EPI_STORE_F32, splits);
                if (rc == 0) launch_splitk_finish(stream, (const float*)workspace, splits, out, ldc, M, N, epi, next);
            } else if (splits > 1)
                rc = launch_tiles_128(stream, A, lda, W, out, ldc, M, N, K, epi, splits, (float*)workspace, next);
            else {
                rc = small && fourwave_takes(epi, out, ldc, N) ? launch_mid(stream, plan.rows, A, lda, W, out, ldc, M, N, K, epi)
                                                               : launch_tiles_128(stream, A, lda, W, out, ldc, M, N, K, epi, 1, nullptr);
                if (rc == 0 && whole) launch_norm_rows(stream, out, ldc, M, N, *next);
            }
        }
        else rc = launch_tiled<128, 128, 64, 1>(stream, A, lda, W, out, ldc, M, N, K, epi);
    }
    if (rc != 0) return -1;
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        llmrs_fail("gemm (mfma): launch failed: %s", hipGetErrorString(e));
        return -1;
    }
    return 1;
}
