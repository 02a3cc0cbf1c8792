// 17 to 64 rows of bfloat16 times a weight whose rows are whole k-blocks (K % 64 == 0): a ring of k-blocks in LDS.
// (part of gemm_mfma.hip)
//
// What bounds the few-row products with this many tokens is neither the weight's bytes nor their latency but the address
// unit in front of the vector cache: an MFMA operand read straight from memory is 16 rows to every 16 lanes, 64 lines an
// instruction instead of 8, and with every block reading the tokens' rows beside its own of the weight (64 rows of 4096: 512 KB
// beside 196 KB of a block of 24 features) those lines, one a clock, took longer than the bytes.  So nothing is
// read that way here: loads straight into LDS (global_load_lds, 8 rows of 128 bytes each) bring whole lines, several stages ahead, and
// the operands come from LDS.  Chunk c of row r lies in slot c ^ (r & 7) of its row: eight lanes' reads hit eight bank groups.
// A block owns (NT - 1) 16 + LAST features and all tokens, a wave one tile of 16 tokens (and with two token tiles every
// other tile of features): sums are whole when the walk ends, nothing is added up between waves.  With gridDim.y > 1 the
// k-blocks are shared out over that many blocks: each writes its 32-bit sums to `partial` [gridDim.y][M][N].
// Measured at 64 rows, operands straight from memory -> from LDS (MI355X, us, with the adding up of parts where there are any):
// 6144 x 4096 25.3 -> 20.2, 4096 x 4096 18.7 -> 15.6, 4096 x 14336 40.6 -> 32.5, 28672 x 4096 54 -> 46, 128256 x 4096 275 -> 222,
// 16384 x 2048 23.8 -> 19.2, 3072 x 2048 12.7 -> 10.0; at 32 rows 28672 x 4096 46.1 -> 44.7, 4096 x 14336 32.4 -> 28.7.
#pragma once
#include "cache_layout.h"
#include "gemm_tile.h"

template <int MT>
constexpr int ring_waves() { return MT == 2 ? 4 : MT; }
template <int MT, int NT, int LAST>
constexpr int ring_stage_bytes(int ksub) { return (((NT - 1) * 16 + LAST) / 8 + 2 * MT) * 1024 * ksub; }

template <int MT, int NT, int LAST, int KSUB, int STAGES>
__global__ __launch_bounds__(64 * ring_waves<MT>()) void gemm_ring_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W, void* __restrict__ out, int lda, int ldc,
                                                                          int M, int N, int K, int epi, float* __restrict__ partial, int rot_feats, QkvEpilogue qe) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char ring_smem[];
    constexpr int WAVES = ring_waves<MT>(), WN = WAVES / MT, TPW = (NT + WN - 1) / WN;     // tiles of features a wave takes at most
    constexpr int BF = (NT - 1) * 16 + LAST, WG = BF / 8, GROUPS = WG + 2 * MT, PER = (GROUPS + WAVES - 1) / WAVES;
    constexpr int STAGE = GROUPS * 1024 * KSUB;
    static_assert((STAGES - 2) * PER * KSUB < 64 && STAGES >= 3, "vmcnt counts to 63");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, g = lane >> 4, mt = wave % MT, wn = wave / MT;
    const int n0 = blockIdx.x * BF;
    // this wave's groups of eight rows (the last one is brought twice or three times where they do not divide: the same bytes)
    const bf16* src[PER];
    int dst[PER];
    {
        const int lrow = lane >> 3, piece = ((lane & 7) ^ lrow) * 8;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int grp = min(wave + i * WAVES, GROUPS - 1);
            dst[i] = grp * 1024;
            src[i] = grp < WG ? W + (size_t)min(n0 + grp * 8 + lrow, N - 1) * K + piece : A + (size_t)min((grp - WG) * 8 + lrow, M - 1) * lda + piece;
        }
    }
    const int nkb = K / 64, share = (nkb + (int)gridDim.y - 1) / (int)gridDim.y, lo = blockIdx.y * share;
    const int cnt = max(min(nkb, lo + share) - lo, 0);                  // this block's k-blocks: [lo, lo + cnt)
    // the walk begins at a place of its own and wraps round, by groups of rot_feats features (see gemm_few.hip)
    const int rot = (cnt > 0 && rot_feats > 0) ? (n0 / rot_feats) % cnt : 0;
    const int steps = (cnt + KSUB - 1) / KSUB;
    auto issue = [&](int s) {
        const int base = (s % STAGES) * STAGE;
#pragma unroll
        for (int ks = 0; ks < KSUB; ++ks) {
            int j = min(s * KSUB + ks, cnt - 1) + rot;
            const int kb = lo + (j >= cnt ? j - cnt : j);
#pragma unroll
            for (int i = 0; i < PER; ++i)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + (size_t)kb * 64),
                                                 (__attribute__((address_space(3))) void*)(ring_smem + __builtin_amdgcn_readfirstlane(base + ks * GROUPS * 1024 + dst[i])), 16, 0, 0);
        }
    };
    f32x4 acc[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // a lane holds token lane % 16 of the wave's tile and features 4 (lane / 16) + r of each of its tiles; out += sum: the old values are
    // asked for ahead of the weights (asked for after them they were a trip to memory more: 1 to 2 % of the products of up to 4096 x 1024)
    const int m = mt * 16 + row;
    const bool adds = partial == nullptr && epi == LLMRS_EPI_ACCUM_F32;
    float old[TPW][4];
    if (adds) {
#pragma unroll
        for (int t = 0; t < TPW; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) old[t][r] = ((const float*)out)[(size_t)min(m, M - 1) * ldc + min(n0 + (wn + t * WN) * 16 + 4 * g + r, N - 1)];
    }
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < steps) issue(s);
    const int off0 = row * 128 + ((g ^ (row & 7)) * 16), off1 = row * 128 + (((4 + g) ^ (row & 7)) * 16);       // a lane's two pieces of a row tile
    for (int s = 0; s < steps; ++s) {
        // stage s has landed when all but the loads of the stages behind it have; behind the barrier every wave's part of it has, and
        // every wave is done with the stage that the next loads go into
        if (s + STAGES - 1 <= steps) wait_vmcnt<(STAGES - 2) * PER * KSUB>(); else wait_vmcnt<0>();
        block_sync_lds();
        if (s + STAGES - 1 < steps) issue(s + STAGES - 1);
        const unsigned char* st = ring_smem + (s % STAGES) * STAGE;
#pragma unroll
        for (int ks = 0; ks < KSUB; ++ks) {
            if (KSUB > 1 && s * KSUB + ks >= cnt) break;
            const unsigned char* ws = st + ks * GROUPS * 1024;
            const unsigned char* xs = ws + WG * 1024 + mt * 2048;
            const bf16x8 x0 = *(const bf16x8*)(xs + off0), x1 = *(const bf16x8*)(xs + off1);
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                const int nt = wn + t * WN;
                if (WN > 1 && nt >= NT) break;
                // (the half of the last tile that is not the block's reads what lies behind: its sums are not used)
                const bf16x8 w0 = *(const bf16x8*)(ws + nt * 2048 + off0), w1 = *(const bf16x8*)(ws + nt * 2048 + off1);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, x0, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, x1, acc[t], 0, 0, 0);
            }
        }
    }
    if (m >= M) return;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const int nt = wn + t * WN, n = n0 + nt * 16 + 4 * g;
        if (nt >= NT || (LAST < 16 && nt == NT - 1 && 4 * g >= LAST)) continue;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[t][r];
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
        } else if (adds) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) ((float*)out)[(size_t)m * ldc + n + r] = old[t][r] + v[r];
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) epilogue_store<bf16>(epi, out, ldc, m, n + r, v[r]);
        }
    }
}
