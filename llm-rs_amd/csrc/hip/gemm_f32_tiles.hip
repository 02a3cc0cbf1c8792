// 32-bit products of many rows on the matrix cores: v_mfma_f32_32x32x2_f32 multiplies and adds in 32-bit (no
// reduced-precision mode).  Needs K % 32 == 0 and 16-byte aligned rows.
//
// The tiles go straight into LDS (global_load_lds_dwordx4), rows of 32 k = 128 bytes, unpadded, with the 16-byte chunk c of
// row r in slot c ^ ((r >> 1) & 7) of its row, as the bfloat16 tiles' are: a lane reads an operand's four k-values as
// one chunk, lanes 0..31 chunk 2 s and lanes 32..63 chunk 2 s + 1 of their row, and MFMA j of step s contracts k = 8 s + j and
// 8 s + 4 + j.  The order of an output's sum depends on K only, so both tile sizes give the same bits.
//
// What bounds it: the matrix cores (a 32-bit MFMA is 64 cycles long: what is read from LDS for it takes a fraction of
// that), where there are blocks enough; so the tile is chosen by how many blocks there are.  Measured (us; before: 128 x 128
// tiles staged through registers, 16 k at a time): 1023 rows 2048 x 8192 704 -> 316 (109 TFLOP/s), 2048 x 2048 188 -> 83,
// 3072 x 2048 194 -> 126, 16384 x 2048 660 -> 591 (116 TFLOP/s of 157 nominal).
#include "gemm_tile.h"

template <int BM, int BN, int WGM, int WGN, int STAGES>
__global__ __launch_bounds__(64 * WGM * WGN) void gemm_f32_dma_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W,
                                                                      void* __restrict__ out, int ldc, int M, int N, int K, int epi) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char f32_smem[];
    constexpr int WAVES = WGM * WGN;
    constexpr int TM = BM / WGM, TN = BN / WGN, FM = TM / 32, FN = TN / 32;
    constexpr int STAGE_BYTES = (BM + BN) * 128;
    constexpr int A_GROUPS = BM / 8 / WAVES, W_GROUPS = BN / 8 / WAVES;   // groups of 8 rows a wave brings in
    constexpr int LOADS = A_GROUPS + W_GROUPS;
    static_assert(A_GROUPS >= 1 && W_GROUPS >= 1, "every wave brings whole groups of 8 rows of both operands");
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int wm = wave / WGN, wn = wave % WGN;
    int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    int lrow = lane >> 3, lslot = lane & 7;
    const float* ga[A_GROUPS];
    const float* gw[W_GROUPS];
#pragma unroll
    for (int i = 0; i < A_GROUPS; ++i) {
        int row = (wave * A_GROUPS + i) * 8 + lrow;
        ga[i] = A + (size_t)min(m0 + row, M - 1) * lda + ((lslot ^ ((row >> 1) & 7)) * 4);
    }
#pragma unroll
    for (int i = 0; i < W_GROUPS; ++i) {
        int row = (wave * W_GROUPS + i) * 8 + lrow;
        gw[i] = W + (size_t)min(n0 + row, N - 1) * K + ((lslot ^ ((row >> 1) & 7)) * 4);
    }
    const int nk = K / 32;
    auto issue = [&](int kt, int stage) {
        unsigned base = __builtin_amdgcn_readfirstlane(stage * STAGE_BYTES + wave * A_GROUPS * 1024);
#pragma unroll
        for (int i = 0; i < A_GROUPS; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(ga[i] + kt * 32),
                                             (__attribute__((address_space(3))) void*)(f32_smem + base + i * 1024), 16, 0, 0);
        unsigned wbase = __builtin_amdgcn_readfirstlane(stage * STAGE_BYTES + BM * 128 + wave * W_GROUPS * 1024);
#pragma unroll
        for (int i = 0; i < W_GROUPS; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(gw[i] + kt * 32),
                                             (__attribute__((address_space(3))) void*)(f32_smem + wbase + i * 1024), 16, 0, 0);
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
        const unsigned char* as = f32_smem + stage * STAGE_BYTES;
        const unsigned char* ws = as + BM * 128;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            f32x4 a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                int row = wm * TM + i * 32 + frow;
                a[i] = *(const f32x4*)(as + row * 128 + (((s * 2 + h) ^ ((row >> 1) & 7)) * 16));
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                int row = wn * TN + j * 32 + frow;
                b[j] = *(const f32x4*)(ws + row * 128 + (((s * 2 + h) ^ ((row >> 1) & 7)) * 16));
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][q], b[j][q], acc[i][j], 0, 0, 0);
        }
        if (kt + STAGES - 1 < nk) wait_vmcnt<(STAGES - 2) * LOADS>(); else wait_vmcnt<0>();
        block_sync_lds();
    }
    static_for<0, FM * FN>([&](auto idx) {
        constexpr int i = decltype(idx)::value / FN, j = decltype(idx)::value % FN;
        int n = n0 + wn * TN + j * 32 + (lane & 31);
        float old[16];
        if (epi == LLMRS_EPI_ACCUM_F32) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                int m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
                old[r] = ((const float*)out)[(size_t)min(m, M - 1) * ldc + min(n, N - 1)];
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            int m = m0 + wm * TM + i * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
            float v = acc[i][j][r];
            if (epi_gated(epi)) {
                float other = swap_neighbours(v);                 // even lane: gate here, up next door
                if (!(lane & 1) && m < M && n + 1 < N) ((float*)out)[(size_t)m * ldc + n / 2] = gated_act(epi, v, other);
            } else if (m < M && n < N) {
                ((float*)out)[(size_t)m * ldc + n] = epi == LLMRS_EPI_ACCUM_F32 ? old[r] + v : v;
            }
        }
    });
}

template <int BM, int BN, int WGM, int WGN, int STAGES>
static int launch_f32_dma(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi) {
    static bool configured = false;
    size_t bytes = (size_t)STAGES * (BM + BN) * 128;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_f32_dma_kernel<BM, BN, WGM, WGN, STAGES>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return llmrs_fail("gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        configured = true;
    }
    dim3 grid(ceil_div(N, BN), ceil_div(M, BM));
    if (grid.y > 65535) return llmrs_fail("gemm: M=%d is too large for one launch", M);
    gemm_f32_dma_kernel<BM, BN, WGM, WGN, STAGES><<<grid, 64 * WGM * WGN, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi);
    return 0;
}

int llmrs_gemm_f32_tiles(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi) {
    // Two forms: 128 x 128 tiles, two blocks to a unit (a third less traffic), and 64 x 64 tiles, four to five to a unit (small
    // grids fill the device, and the last round costs less).  Time in units of one 128 x 128 block alone on its unit
    // (at K = 2048: 138 us): two on a unit take 2.13, 64 x 64 blocks 0.00118 each once they are more than two to a unit
    // and 0.6 for a unit's two.
    const int cus = llmrs_compute_units();
    const long big = (long)ceil_div(M, 128) * ceil_div(N, 128), small = (long)ceil_div(M, 64) * ceil_div(N, 64);
    const long last = big % (2L * cus);
    const double big_time = 2.13 * (double)(big / (2L * cus)) + (last == 0 ? 0.0 : last <= cus ? 1.0 : 2.13);
    const double small_time = small <= 2L * cus ? 0.6 : 0.302 / cus * (double)small;
    // (64-row tiles of more rows than a grid has room for: the larger ones)
    if (big_time <= small_time || ceil_div(M, 64) > 65535) return launch_f32_dma<128, 128, 2, 2, 2>(stream, A, lda, W, out, ldc, M, N, K, epi);
    // (a block alone on its unit: three k-tiles in LDS; 45 against 53 us at 2048 x 2048.  With more to a unit the room is
    // better given to another block: 83 against 89.)
    if (small <= cus) return launch_f32_dma<64, 64, 2, 2, 3>(stream, A, lda, W, out, ldc, M, N, K, epi);
    return launch_f32_dma<64, 64, 2, 2, 2>(stream, A, lda, W, out, ldc, M, N, K, epi);
}
