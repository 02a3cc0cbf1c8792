// 32-bit products of many rows on the matrix cores: v_mfma_f32_16x16x4_f32 multiplies and adds in 32-bit (no
// reduced-precision mode).  Needs K % 32 == 0 and 16-byte aligned rows.
//
// The tiles go straight into LDS (global_load_lds_dwordx4), rows of 32 k = 128 bytes, unpadded, with the 16-byte chunk c of
// row r in slot c ^ ((r >> 1) & 7) of its row, as the bfloat16 tiles' are: a lane reads an operand's four k-values as
// one chunk, lanes 16 g .. 16 g + 15 chunk 4 s + g of their row, and MFMA j of step s contracts k = 16 s + 4 g + j over g.  The
// order of an output's sum depends on K only, so all tile sizes give the same bits.
//
// What bounds it: the matrix cores (a 32-bit MFMA is 32 cycles long: what is read from LDS for it takes a fraction of
// that), as far as the loop leaves them no gaps.  A step's operands are asked for while the step before is multiplied, across the barrier
// too, and the loads of a k-tile go out one by one between its MFMAs: asked for together they hold the wave at the
// address unit (16 cycles each, 16 to 48 of them between the four waves) while its matrix core is idle.  Features are the rows of the
// MFMAs and tokens their columns, so a lane ends with four consecutive features of a token: 16 bytes to store, gated pairs in one lane.
// Measured (us; operands read where they are used and a k-tile's loads all at once, on v_mfma_f32_32x32x2_f32, then now): 1023 rows
// 16384 x 2048 gated 518 -> 493 (139 TFLOP/s; these MFMAs alone reach 138-150 as the clock follows their power, 157 is nominal), 2048 x 8192
// 283 -> 269, 2048 x 2048 79 -> 76, 3072 x 2048 108 -> 101; 512 rows 28672 x 4096 gated 1088 -> 903 and 2048 rows 3568 -> 3327 (there
// also the order of the tiles, tile_of_block).  Errors against 64 bits are the same (1023 x 2048 x 8192 1.64e-6 and 1.61e-6 of the result's size).
#include "gemm_tile.h"
#include <algorithm>

template <int BM, int BN, int STAGES>
__global__ __launch_bounds__(256, 2) void gemm_f32_dma_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W,
                                                           void* __restrict__ out, int ldc, int M, int N, int K, int epi) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char f32_smem[];
    constexpr int WAVES = 4, TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16;
    constexpr int STAGE_BYTES = (BM + BN) * 128;
    constexpr int LOADS = (BM + BN) / 8 / WAVES;       // groups of 8 rows a wave brings in
    static_assert(BM % 32 == 0 && BN % 32 == 0 && LOADS % 2 == 0, "every wave brings whole groups of 8 rows, half of them in either step");
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int wm = wave / 2, wn = wave % 2;
    int tile_row, tile_column;
    tile_of_block(K, tile_row, tile_column);
    int m0 = tile_row * BM, n0 = tile_column * BN;
    int lrow = lane >> 3, lslot = lane & 7;
    const float* from[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        int row = (wave * LOADS + i) * 8 + lrow, chunk = (lslot ^ ((row >> 1) & 7)) * 4;
        from[i] = row < BM ? A + (size_t)min(m0 + row, M - 1) * lda + chunk : W + (size_t)min(n0 + row - BM, N - 1) * K + chunk;
    }
    const int nk = K / 32;
    // loads FIRST to LAST - 1 of this wave's part of k-tile kt (past the end: the last tile once more, never used)
    auto ask = [&](int kt, int stage, auto firstc, auto lastc) {
        unsigned base = __builtin_amdgcn_readfirstlane(stage * STAGE_BYTES + wave * LOADS * 1024);
        kt = min(kt, nk - 1);
#pragma unroll
        for (int i = decltype(firstc)::value; i < decltype(lastc)::value; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from[i] + kt * 32),
                                             (__attribute__((address_space(3))) void*)(f32_smem + base + i * 1024), 16, 0, 0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using Half = std::integral_constant<int, LOADS / 2>;
    using All = std::integral_constant<int, LOADS>;
    f32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int frow = lane & 15, g = lane >> 4;
    unsigned offa[2], offb[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        unsigned chunk = (unsigned)(((s * 4 + g) ^ ((frow >> 1) & 7)) * 16);
        offa[s] = (wm * TM + frow) * 128 + chunk;
        offb[s] = (BM + wn * TN + frow) * 128 + chunk;
    }
    f32x4 a[2][FM], b[2][FN];
    auto read = [&](const unsigned char* st, auto sc) {
        constexpr int s = decltype(sc)::value;
#pragma unroll
        for (int i = 0; i < FM; ++i) a[s][i] = *(const f32x4*)(st + offa[s] + i * 16 * 128);
#pragma unroll
        for (int j = 0; j < FN; ++j) b[s][j] = *(const f32x4*)(st + offb[s] + j * 16 * 128);
    };
    auto mult = [&](auto sc) {
        constexpr int s = decltype(sc)::value;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[s][j][q], a[s][i][q], acc[i][j], 0, 0, 0);
    };
    // a step's operands one by one with an MFMA after each, then its loads, evenly over the MFMAs that are left
    auto order = [] {
        constexpr int MULTS = 4 * FM * FN, READS = FM + FN, N_LOADS = LOADS / 2, apart = (MULTS - READS) / N_LOADS > 0 ? (MULTS - READS) / N_LOADS : 1;
        static_for<0, READS>([](auto) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        });
        static_for<0, N_LOADS>([](auto) {
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, apart, 0);
        });
        __builtin_amdgcn_sched_group_barrier(0x008, MULTS, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int p = 0; p < STAGES - 1; ++p) ask(p, p, I0{}, All{});
    wait_vmcnt<(STAGES - 2) * LOADS>();
    __syncthreads();
    // k-tile kt lies in stage `at`; k-tile kt + STAGES - 1 goes where kt - 1 was, whose last reads every wave finished before the barrier
    int at = 0, into = STAGES - 1;
    auto k_tile = [&](int kt, auto not_first) {
        const unsigned char* st = f32_smem + at * STAGE_BYTES;
        read(st, I0{});
        ask(kt + STAGES - 1, into, I0{}, Half{});
        if constexpr (decltype(not_first)::value) mult(I1{});
        order();
        read(st, I1{});
        ask(kt + STAGES - 1, into, Half{}, All{});
        mult(I0{});
        order();
        wait_vmcnt<(STAGES - 2) * LOADS>();
        block_sync_lds();
        __builtin_amdgcn_sched_barrier(0);
        at = at + 1 == STAGES ? 0 : at + 1;
        into = into + 1 == STAGES ? 0 : into + 1;
    };
    k_tile(0, std::false_type{});
    for (int kt = 1; kt < nk; ++kt) k_tile(kt, std::true_type{});
    mult(I1{});
    wait_vmcnt<0>();               // (no load into LDS is left on its way: the waves' bands go there now)
    __syncthreads();
    const int m_first = m0 + wm * TM, n_first = n0 + wn * TN;
    if (epi_gated(epi))
        bands_to_f32<FM, FN, true>(f32_smem + wave * (16 * (TN * 2 + 16)), (float*)out, ldc, M, N / 2, m_first, n_first / 2, false, [&](auto ic, auto jc) {
            const f32x4 v = acc[decltype(ic)::value][decltype(jc)::value];
            return f32x4{gated_act(epi, v[0], v[1]), gated_act(epi, v[2], v[3]), 0.0f, 0.0f};
        });
    else
        bands_to_f32<FM, FN, false>(f32_smem + wave * (16 * (TN * 4 + 16)), (float*)out, ldc, M, N, m_first, n_first, epi == LLMRS_EPI_ACCUM_F32,
                                    [&](auto ic, auto jc) { return acc[decltype(ic)::value][decltype(jc)::value]; });
}

template <int BM, int BN, int STAGES>
static int launch_f32_dma(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi) {
    static bool configured = false;
    size_t bytes = (size_t)STAGES * (BM + BN) * 128;
    if (!configured) {
        hipError_t e = hipFuncSetAttribute((const void*)gemm_f32_dma_kernel<BM, BN, STAGES>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return llmrs_fail("gemm: cannot reserve %zu bytes of LDS: %s", bytes, hipGetErrorString(e));
        configured = true;
    }
    dim3 grid(ceil_div(N, BN), ceil_div(M, BM));
    if (grid.y > 65535) return llmrs_fail("gemm: M=%d is too large for one launch", M);
    gemm_f32_dma_kernel<BM, BN, STAGES><<<grid, 256, bytes, stream>>>(A, lda, W, out, ldc, M, N, K, epi);
    return 0;
}

int llmrs_gemm_f32_tiles(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi) {
    // Two forms: 128 x 128 tiles, two blocks to a unit, and 64 x 64 tiles, three to a unit (small grids fill the device, and the last
    // round costs less).  Time in units of one 128 x 128 block alone on its unit (at K = 2048: 137 us): two on a unit take 1.79; 64 x 64
    // blocks 0.238 each, a unit's first 0.31 and its first two 0.56.  (Tiles of 256 x 128, a block to a unit, take as long as two of 128 x 128.)
    const int cus = llmrs_compute_units();
    const long big = (long)ceil_div(M, 128) * ceil_div(N, 128), small = (long)ceil_div(M, 64) * ceil_div(N, 64);
    const long last = big % (2L * cus);
    const double big_time = 1.79 * (double)(big / (2L * cus)) + (last == 0 ? 0.0 : last <= cus ? 1.0 : 1.79);
    const double small_time = std::max(small <= cus ? 0.31 : 0.56, 0.238 / cus * (double)small);
    // (64-row tiles of more rows than a grid has room for: the larger ones)
    if (big_time <= small_time || ceil_div(M, 64) > 65535) return launch_f32_dma<128, 128, 2>(stream, A, lda, W, out, ldc, M, N, K, epi);
    return launch_f32_dma<64, 64, 3>(stream, A, lda, W, out, ldc, M, N, K, epi);
}
