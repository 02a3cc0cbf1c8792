// The plain product: 64x64 tiles through LDS, 32-bit FMA, k in ascending order.
// With the 32-bit matrix-core tiles (here and in gemm_f32_tiles.hip), the products of few rows (gemm_few.hip) and the kernels
// of some more below it is the whole 32-bit path (nothing here rounds its inputs) and the bfloat16 fallback for shapes
// the bfloat16 MFMA kernels refuse.  Within each kernel the order of
// the sum for an output depends on K only (and on the weight's shape), so a row's result does not depend on the
// row's place in the batch or on its tile; which kernel runs depends on M and the shape, so across those
// ranges results differ by rounding.
// Reference: gemm_f32 accumulates in 32-bit the same way (shaders/ops.metal:1053-1079).
#include "gemm.h"

#define TILE 64
#define TILE_K 16

template <class T>
__global__ __launch_bounds__(256) void gemm_simple_kernel(const T* __restrict__ A, int lda,
                                                          const T* __restrict__ W, void* __restrict__ out, int ldc,
                                                          int M, int N, int K, int epi) {
    __shared__ float As[TILE_K][TILE + 4];
    __shared__ float Ws[TILE_K][TILE + 4];
    int tid = threadIdx.x;
    int m0 = blockIdx.y * TILE, n0 = blockIdx.x * TILE;
    int ty = tid / 16, tx = tid % 16;
    int lrow = tid / 4, lk = (tid % 4) * 4;  // this thread stages 4 k-values of one row of each tile
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += TILE_K) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int k = k0 + lk + i;
            int am = m0 + lrow, wn = n0 + lrow;
            As[lk + i][lrow] = (am < M && k < K) ? to_f32(A[(size_t)am * lda + k]) : 0.0f;
            Ws[lk + i][lrow] = (wn < N && k < K) ? to_f32(W[(size_t)wn * K + k]) : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < TILE_K; ++kk) {
            float a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = Ws[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        int m = m0 + ty * 4 + i;
        if (m >= M) continue;
        if (epi_gated(epi)) {
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                int n = n0 + tx * 4 + j;
                if (n + 1 < N) ((T*)out)[(size_t)m * ldc + n / 2] = from_f32<T>(gated_act(epi, acc[i][j], acc[i][j + 1]));
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int n = n0 + tx * 4 + j;
                if (n < N) epilogue_store<T>(epi, out, ldc, m, n, acc[i][j]);
            }
        }
    }
}

// 32-bit products on the matrix cores for rows that cannot be read in 16-byte pieces of whole 32-k blocks (gemm_f32_tiles.hip
// and the few-row kernel below take the others): v_mfma_f32_32x32x2_f32 multiplies and adds in 32-bit (no
// reduced-precision mode), k in ascending order, so an output's sum depends on K only here too.
// 128 x 128 tiles of four waves (64 x 64 each), k in steps of 16 through two LDS buffers; the next
// step's rows are on their way to registers while this step is multiplied.  Any M, N, K: rows and
// k beyond the edges are read as zeros.
typedef float f32x16_t __attribute__((ext_vector_type(16)));
#define F32_BK 16
#define F32_LD (F32_BK + 1)      // LDS row stride in floats: lanes of an operand read (32 rows, one k each) hit distinct banks
__global__ __launch_bounds__(256) void gemm_f32_mfma_kernel(const float* __restrict__ A, int lda,
                                                            const float* __restrict__ W, void* __restrict__ out, int ldc,
                                                            int M, int N, int K, int epi) {
    __shared__ float As[2][128 * F32_LD];
    __shared__ float Ws[2][128 * F32_LD];
    int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int wm = wave >> 1, wn = wave & 1;
    int m0 = blockIdx.y * 128, n0 = blockIdx.x * 128;
    // staging: thread t brings 4 consecutive k of rows (t / 4) and (t / 4 + 64) of each tile
    int srow = tid >> 2, sk = (tid & 3) * 4;
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0;
    float ra[2][4], rw[2][4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            int am = m0 + srow + 64 * h, wn_ = n0 + srow + 64 * h, k = k0 + sk;
            const float* ap = A + (size_t)min(am, M - 1) * lda + k;
            const float* wp = W + (size_t)min(wn_, N - 1) * K + k;
            if (vec && k + 3 < K) {
                load4(ap, ra[h]);
                load4(wp, rw[h]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    ra[h][j] = k + j < K ? ap[j] : 0.0f;
                    rw[h][j] = k + j < K ? wp[j] : 0.0f;
                }
            }
            if (am >= M)
#pragma unroll
                for (int j = 0; j < 4; ++j) ra[h][j] = 0.0f;
            if (wn_ >= N)
#pragma unroll
                for (int j = 0; j < 4; ++j) rw[h][j] = 0.0f;
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                As[buf][(srow + 64 * h) * F32_LD + sk + j] = ra[h][j];
                Ws[buf][(srow + 64 * h) * F32_LD + sk + j] = rw[h][j];
            }
    };
    f32x16_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    int nk = (K + F32_BK - 1) / F32_BK;
    fetch(0);
    stage(0);
    __syncthreads();
    int frow = lane & 31, fk = lane >> 5;
    for (int kt = 0; kt < nk; ++kt) {
        int buf = kt & 1;
        if (kt + 1 < nk) fetch((kt + 1) * F32_BK);
        const float* as = As[buf] + (wm * 64 + frow) * F32_LD + fk;
        const float* ws = Ws[buf] + (wn * 64 + frow) * F32_LD + fk;
#pragma unroll
        for (int ks = 0; ks < F32_BK / 2; ++ks) {
            float a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = as[i * 32 * F32_LD + ks * 2];
#pragma unroll
            for (int j = 0; j < 2; ++j) b[j] = ws[j * 32 * F32_LD + ks * 2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) stage(buf ^ 1);        // the other buffer's readers finished before the last barrier
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            int n = n0 + wn * 64 + j * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                float v = acc[i][j][r];
                if (epi_gated(epi)) {
                    float other = __shfl_xor(v, 1, 64);   // even lane: gate here, up next door
                    if (!(lane & 1) && m < M && n + 1 < N)
                        ((float*)out)[(size_t)m * ldc + n / 2] = gated_act(epi, v, other);
                } else if (m < M && n < N) {
                    epilogue_store<float>(epi, out, ldc, m, n, v);
                }
            }
        }
}

// A few tokens (decoding): a wave for each pair of weight rows, every weight read once.
// Lanes stride over k, four elements at a time, and each keeps one 32-bit sum per token and
// row; the lanes' sums are added by a butterfly.  The order depends on K only.
#define GEMV_MAX_M 8
// VEC: K % 4 == 0 and every row starts on a multiple of four elements' size, so a lane's four
// elements come in one load and none of them lies past K.  RW weight rows per wave (even): the
// tokens' rows are read once for all of them.  The sums are the same whatever VEC and RW are.
template <class T, bool VEC, int RW>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const T* __restrict__ A, int lda, const T* __restrict__ W,
                                                        void* __restrict__ out, int ldc, int M, int N, int K, int epi) {
    int lane = threadIdx.x & 63;
    int n = RW * (blockIdx.x * 4 + (threadIdx.x >> 6));
    if (n >= N) return;
    const T* w[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) w[r] = W + (size_t)min(n + r, N - 1) * K;
    float acc[RW][GEMV_MAX_M] = {};
#pragma unroll 2
    for (int k = lane * 4; k < K; k += 256) {
        float a[RW][4];
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            if constexpr (VEC) {
                load4(w[r] + k, a[r]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) a[r][j] = k + j < K ? to_f32(w[r][k + j]) : 0.0f;
            }
        }
#pragma unroll
        for (int m = 0; m < GEMV_MAX_M; ++m) {
            if (m >= M) break;
            const T* x = A + (size_t)m * lda + k;
            float xv[4];
            if constexpr (VEC) {
                load4(x, xv);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) xv[j] = k + j < K ? to_f32(x[j]) : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int r = 0; r < RW; ++r) acc[r][m] = fmaf(a[r][j], xv[j], acc[r][m]);
        }
    }
#pragma unroll
    for (int m = 0; m < GEMV_MAX_M; ++m) {
        if (m >= M) break;
        float v[RW];
#pragma unroll
        for (int r = 0; r < RW; ++r) v[r] = wave_sum(acc[r][m]);
        if (lane != 0) continue;
#pragma unroll
        for (int r = 0; r < RW; r += 2) {
            if (epi_gated(epi)) {
                if (n + r + 1 < N) ((T*)out)[(size_t)m * ldc + (n + r) / 2] = from_f32<T>(gated_act(epi, v[r], v[r + 1]));
            } else {
                if (n + r < N) epilogue_store<T>(epi, out, ldc, m, n + r, v[r]);
                if (n + r + 1 < N) epilogue_store<T>(epi, out, ldc, m, n + r + 1, v[r + 1]);
            }
        }
    }
}

// 33 tokens and more in 32-bit on the matrix cores (up to 32: gemm_few.hip, but for 17 to 32 on wide weights with the shortest rows, which
// come here): v_mfma_f32_16x16x4_f32 multiplies and adds in
// 32-bit (no reduced-precision mode).  The weight's rows are the A operand, read once for every 16 MT tokens, 16 bytes a
// lane (lane l: feature l % 16 of a tile, the four k-values 4 (l / 16) .. + 3 of a group of 16); the tokens' rows are the B
// operand, read the same way once for all of a block's NT feature tiles.  An MFMA contracts the four k-values that the
// four lane groups hold in the same place of their loads.  A block's NW waves take the 32-wide k-blocks in turn, U of them
// with all loads asked for before the first product, and add their sums through LDS in wave order.  C: lane l holds token
// l % 16 and features 4 (l / 16) + r.  Needs K % 32 == 0 and 16-byte aligned rows.
// rot_feats > 0: neighbouring groups of that many features begin their walk along k at different k-blocks and wrap
// round.  Rows are a multiple of the memory channels' interleave apart, so blocks in step would all ask the same few
// channels at once.  What bounds it: the weights' bytes, and beside them the tokens' rows, which every block reads again.
typedef float f32x4_t __attribute__((ext_vector_type(4)));
template <int MT, int NT, int NW, int U>
__global__ __launch_bounds__(NW * 64) void gemm_f32_skinny_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W,
                                                                  void* __restrict__ out, int ldc, int M, int N, int K, int epi, int rot_feats) {
    extern __shared__ __attribute__((aligned(16))) float f32_skinny_red[];       // [NW][MT][NT][4][64]
    float* red = f32_skinny_red;
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int row = lane & 15, g = lane >> 4;
    int n0 = blockIdx.x * NT * 16, m0 = blockIdx.y * MT * 16;
    const float* wp[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wp[nt] = W + (size_t)min(n0 + nt * 16 + row, N - 1) * K + 4 * g;
    const float* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) xp[mt] = A + (size_t)min(m0 + mt * 16 + row, M - 1) * lda + 4 * g;
    f32x4_t acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int nkb = K / 32;
    const int rot = rot_feats > 0 ? (int)((unsigned)(n0 / rot_feats) * 37u % (unsigned)nkb) : 0;
    auto turn = [&](int j) { int x = j + rot; return (x >= nkb ? x - nkb : x) * 32; };
    auto products = [&](const f32x4_t (&w)[NT][2], const f32x4_t (&x)[MT][2]) {
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
                        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[nt][half][j], x[mt][half][j], acc[mt][nt], 0, 0, 0);
    };
    auto ask = [&](f32x4_t (&w)[NT][2], f32x4_t (&x)[MT][2], int k) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) { w[nt][0] = *(const f32x4_t*)(wp[nt] + k); w[nt][1] = *(const f32x4_t*)(wp[nt] + k + 16); }
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) { x[mt][0] = *(const f32x4_t*)(xp[mt] + k); x[mt][1] = *(const f32x4_t*)(xp[mt] + k + 16); }
    };
    int kb = wave;
    for (; kb + (U - 1) * NW < nkb; kb += U * NW) {
        f32x4_t w[U][NT][2], x[U][MT][2];
#pragma unroll
        for (int u = 0; u < U; ++u) ask(w[u], x[u], turn(kb + u * NW));
        __builtin_amdgcn_sched_barrier(0);   // keep the round's loads together, ahead of its products
#pragma unroll
        for (int u = 0; u < U; ++u) products(w[u], x[u]);
    }
    for (; kb < nkb; kb += NW) {
        f32x4_t w[NT][2], x[MT][2];
        ask(w, x, turn(kb));
        products(w, x);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[(((wave * MT + mt) * NT + nt) * 4 + r) * 64 + lane] = acc[mt][nt][r];
    __syncthreads();
    // the block's tiles are shared out over its waves; each is summed over the waves in order
    for (int tile = wave; tile < MT * NT; tile += NW) {
        int mt = tile / NT, nt = tile % NT;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float s = 0.0f;
#pragma unroll
            for (int w2 = 0; w2 < NW; ++w2) s += red[(((w2 * MT + mt) * NT + nt) * 4 + r) * 64 + lane];
            v[r] = s;
        }
        int m = m0 + mt * 16 + row, n = n0 + nt * 16 + 4 * g;
        if (m >= M) continue;
        if (epi_gated(epi)) {
#pragma unroll
            for (int r = 0; r < 4; r += 2)
                if (n + r + 1 < N) ((float*)out)[(size_t)m * ldc + (n + r) / 2] = gated_act(epi, v[r], v[r + 1]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) epilogue_store<float>(epi, out, ldc, m, n + r, v[r]);
        }
    }
}

template <int MT, int NT, int NW, int U>
static void launch_f32_skinny(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi, int rot_feats = 0) {
    constexpr size_t bytes = (size_t)NW * MT * NT * 4 * 64 * sizeof(float);
    static_assert(bytes <= 64 * 1024, "the waves' sums must fit in the LDS a block may ask for");
    static bool configured = false;
    if (!configured) {
        (void)hipFuncSetAttribute((const void*)gemm_f32_skinny_kernel<MT, NT, NW, U>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        configured = true;
    }
    gemm_f32_skinny_kernel<MT, NT, NW, U><<<dim3(ceil_div(N, NT * 16), ceil_div(M, MT * 16)), NW * 64, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi, rot_feats);
}

// The kernel above, in the form that the product's shape asks for; false: the tiles take it.
static bool launch_f32_few_rows(hipStream_t stream, const float* a, int lda, const float* w, void* out, int ldc, int M, int N, int K, int epi) {
    const int cus = llmrs_compute_units();
    // Blocks of 32 tokens with the fewest features that still make one round of the compute units.  Where even
    // 64 features to a block make more, the tiles take over, but for up to 32 tokens, whose weights are read once here.
    // (us, this kernel / tiles: 64 rows 3072 x 2048 19 / 45, 16384 x 2048 66 / 48; 100 rows 2048 x 2048 19 / 45; 200 rows 2048 x 2048 29 / 45, 3072 x 2048 58 / 46)
    const long rows = ceil_div(M, 32);
    if (rows * ceil_div(N, 16) <= cus) launch_f32_skinny<2, 1, 4, 4>(stream, a, lda, w, out, ldc, M, N, K, epi, 64);
    else if (rows * ceil_div(N, 32) <= cus) launch_f32_skinny<2, 2, 4, 2>(stream, a, lda, w, out, ldc, M, N, K, epi, 64);
    else if (rows * ceil_div(N, 64) <= cus || M <= 32) launch_f32_skinny<2, 4, 4, 2>(stream, a, lda, w, out, ldc, M, N, K, epi, 64);
    else return false;
    return true;
}

// ---- the slots of the clamped gated epilogue's constants -------------------------------------------------------------
// A set of constants (limit, alpha, cubic, up_add) gets a slot the first time a feed-forward asks for it on a device (when it takes its weights:
// never inside a recording); the slot is written in every source file's table and the stream is waited for, so every
// later product on any stream finds it.  The same set on the same device gets the same slot again.
#include <mutex>
#include <vector>
GluClampTable* llmrs_glu_clamp_tables;               // (null before the first file's table is put on it: no constructor runs for it)
extern "C" int llmrs_glu_clamp_table_count() {
    int n = 0;
    for (const GluClampTable* table = llmrs_glu_clamp_tables; table != nullptr; table = table->next) ++n;
    return n;
}
struct GluSlot { int device; GluClamp p; };
static std::mutex glu_mutex;
static std::vector<GluSlot> glu_slots;
static int glu_clamp_slots_taken() {
    std::lock_guard<std::mutex> lock(glu_mutex);
    return (int)glu_slots.size();
}
extern "C" int llmrs_glu_clamp_slot(hipStream_t stream, float limit, float alpha, float cubic, float up_add) {
    if (!(limit > 0.0f)) { llmrs_fail("glu_clamp_slot: the limit must be positive, got %g", limit); return -1; }
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) { llmrs_fail("glu_clamp_slot: no current device"); return -1; }
    std::lock_guard<std::mutex> lock(glu_mutex);
    for (size_t i = 0; i < glu_slots.size(); ++i)
        if (glu_slots[i].device == device && glu_slots[i].p.limit == limit && glu_slots[i].p.alpha == alpha && glu_slots[i].p.cubic == cubic &&
            glu_slots[i].p.up_add == up_add) return (int)i;
    if (glu_slots.size() >= LLMRS_GLU_SLOTS) { llmrs_fail("glu_clamp_slot: more than %d different sets of constants", LLMRS_GLU_SLOTS); return -1; }
    int slot = (int)glu_slots.size();
    GluClamp p{limit, alpha, cubic, up_add};
    for (const GluClampTable* table = llmrs_glu_clamp_tables; table != nullptr; table = table->next) table->store(stream, slot, p);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) { llmrs_fail("glu_clamp_slot: %s", hipGetErrorString(e)); return -1; }
    glu_slots.push_back(GluSlot{device, p});
    return slot;
}

// A: [M, K] with row stride lda; W: [N, K] dense; out: row stride ldc (elements of
// its own type; for SWIGLU the output has N/2 columns).  workspace: optional device
// memory (16 * 64 * N * 4 bytes is always enough) for products that split K over blocks.
// scale_sumsq (with its parts and eps): a norm left to this product, see RowScale in gemm.h.  next_sumsq (with next_y,
// its row stride and the next norm's weight): what the += epilogue leaves for the norm that follows, see NextNorm.
// Both null in the ordinary case; otherwise the product must be one llmrs_gemm_defers_norm(M, N, K) accepts, in
// bfloat16 or (llmrs_gemm_f32_defers_norm) in 32-bit on the matrix cores, or the call fails.
extern "C" int llmrs_gemm(hipStream_t stream, int dtype, const void* A, int lda, const void* W, void* out, int ldc,
                          int M, int N, int K, int epi, void* workspace, size_t workspace_bytes, int allow_mfma,
                          const float* scale_sumsq, int scale_parts, float scale_eps, float* next_sumsq, void* next_y,
                          int next_ldy, const float* next_weight, float next_eps) {
    LLMRS_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
    LLMRS_REQUIRE(lda >= K, "gemm: row stride %d of A is shorter than K=%d", lda, K);
    LLMRS_REQUIRE((epi >= 0 && epi <= 3) || (epi >= LLMRS_EPI_GLU_CLAMP && epi < LLMRS_EPI_GLU_CLAMP + glu_clamp_slots_taken()),
                  "gemm: unknown epilogue %d (a clamped gated epilogue is %d + a slot that llmrs_glu_clamp_slot gave)", epi, (int)LLMRS_EPI_GLU_CLAMP);
    if (epi_gated(epi)) {
        LLMRS_REQUIRE(N % 2 == 0, "gemm: the gate/up epilogue needs an even N, got %d", N);
        LLMRS_REQUIRE(ldc >= N / 2, "gemm: row stride %d of out is shorter than N/2=%d", ldc, N / 2);
    } else {
        LLMRS_REQUIRE(ldc >= N, "gemm: row stride %d of out is shorter than N=%d", ldc, N);
    }
    if (M == 0) return 0;
    if (dtype == LLMRS_BF16 && allow_mfma) {
        RowScale rs{scale_sumsq, scale_parts, scale_eps};
        NextNorm nn{next_sumsq, next_y, next_ldy, next_weight, next_eps};
        int took = llmrs_gemm_bf16_mfma(stream, (const bf16*)A, lda, (const bf16*)W, out, ldc, M, N, K, epi, workspace,
                                        workspace_bytes, nullptr, scale_sumsq ? &rs : nullptr, next_y ? &nn : nullptr);
        if (took != 0) return took < 0 ? -1 : 0;
    }
    const bool f32_cores = dtype == LLMRS_F32 && allow_mfma && K % 32 == 0 && lda % 4 == 0 && ((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0;
    const bool plain = scale_sumsq == nullptr && next_y == nullptr;
    // One or two tokens: the walk below, whose error is the smaller one for K over 128 and under 1024 and which is at least as fast, but for
    // longer rows of narrow weights and of wide ones and the longest rows of those between (1 row, walk / few rows' kernel, us: 512 x 1536 4.8 /
    // 5.4, 2048 x 2048 7.8 / 6.1, 2048 x 8192 23 / 14.6, 4096 x 4096 14.6 / 14.5, 4608 x 1536 7.5 / 10.2, 6144 x 4096 20.0 / 22.1, 9216 x 5120
    // 38.3 / 39.8, 13824 x 5120 56.7 / 52.2; from 65536 on no difference.  2 rows: 1024 x 1024 5.5 / 4.7, 9216 x 5120 41.6 / 40.8, 11008 x 128
    // 4.7 / 3.8, 11008 x 3584 33.9 / 30.1).
    const bool walk = plain && M <= 2 && (N >= 65536 || (N <= 4096 ? K < 1024 || (M == 1 && N <= 1536 && K < 2048)
                                                        : N > 10240 ? K < 2048 : K < 5120 || (M == 1 && N > 8192))) && !(M == 2 && K <= 128 && N < 65536);
    // (17 to 32 on wide weights with the shortest rows with gemm_f32_skinny_kernel: 65536 x 128 16.1 against 19.8 us; from rows of 256 on there is
    // no difference, and the longer ones gain)
    if (f32_cores && M <= 32 && !walk && !(plain && M > 16 && N >= 16384 && K < 256)) {
        LLMRS_REQUIRE(plain || M <= 16, "gemm: a deferred norm needs the matrix-core kernels for few rows (M=%d N=%d K=%d)", M, N, K);
        RowScale rs{scale_sumsq, scale_parts, scale_eps};
        NextNorm nn{next_sumsq, next_y, next_ldy, next_weight, 0.0f};
        if (llmrs_gemm_few_f32(stream, (const float*)A, lda, (const float*)W, out, ldc, M, N, K, epi, nullptr, scale_sumsq ? &rs : nullptr,
                               next_y ? &nn : nullptr) < 0) return -1;
        LLMRS_LAUNCH_CHECK("gemm");
        return 0;
    }
    LLMRS_REQUIRE(plain, "gemm: a deferred norm needs the matrix-core kernels for few rows (M=%d N=%d K=%d)", M, N, K);
    if (f32_cores && M > 2) {
        if (!launch_f32_few_rows(stream, (const float*)A, lda, (const float*)W, out, ldc, M, N, K, epi) &&
            llmrs_gemm_f32_tiles(stream, (const float*)A, lda, (const float*)W, out, ldc, M, N, K, epi) != 0) return -1;
        LLMRS_LAUNCH_CHECK("gemm");
        return 0;
    }
    if (M <= GEMV_MAX_M) {
        size_t elt = dtype == LLMRS_F32 ? sizeof(float) : sizeof(bf16);
        bool vec = K % 4 == 0 && lda % 4 == 0 && (uintptr_t)A % (4 * elt) == 0 && (uintptr_t)W % (4 * elt) == 0;
        // four weight rows per wave once several tokens share them, if that leaves six waves or more
        // for each compute unit (measured in 32-bit at 8 tokens: 28672 x 4096 130 -> 100 us; 4096 rows are
        // better off with two, 49 against 56 us)
        bool four = M > 2 && N >= 24 * llmrs_compute_units();
        int blocks = ceil_div(N, four ? 16 : 8);
#define ROWS(T, V) do { if (four) gemm_rows_kernel<T, V, 4><<<blocks, 256, 0, stream>>>((const T*)A, lda, (const T*)W, out, ldc, M, N, K, epi); \
                        else gemm_rows_kernel<T, V, 2><<<blocks, 256, 0, stream>>>((const T*)A, lda, (const T*)W, out, ldc, M, N, K, epi); } while (0)
        if (dtype == LLMRS_F32) { if (vec) ROWS(float, true); else ROWS(float, false); }
        else if (dtype == LLMRS_BF16) { if (vec) ROWS(bf16, true); else ROWS(bf16, false); }
        else return llmrs_fail("gemm: unknown dtype %d", dtype);
#undef ROWS
        LLMRS_LAUNCH_CHECK("gemm");
        return 0;
    }
    dim3 grid(ceil_div(N, TILE), ceil_div(M, TILE));
    LLMRS_REQUIRE(grid.y <= 65535, "gemm: M=%d is too large for one launch", M);
    if (dtype == LLMRS_F32 && allow_mfma && M > 16) {
        dim3 g128(ceil_div(N, 128), ceil_div(M, 128));
        LLMRS_REQUIRE(g128.y <= 65535, "gemm: M=%d is too large for one launch", M);
        gemm_f32_mfma_kernel<<<g128, 256, 0, stream>>>((const float*)A, lda, (const float*)W, out, ldc, M, N, K, epi);
    } else if (dtype == LLMRS_F32)
        gemm_simple_kernel<float><<<grid, 256, 0, stream>>>((const float*)A, lda, (const float*)W, out, ldc, M, N, K, epi);
    else if (dtype == LLMRS_BF16)
        gemm_simple_kernel<bf16><<<grid, 256, 0, stream>>>((const bf16*)A, lda, (const bf16*)W, out, ldc, M, N, K, epi);
    else
        return llmrs_fail("gemm: unknown dtype %d", dtype);
    LLMRS_LAUNCH_CHECK("gemm");
    return 0;
}
