// What the matrix-core products' tile loops and epilogues share (gemm_mfma.hip, expert_gemm.hip).
#pragma once
#include "cache_layout.h"
#include "gemm.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// The value the neighbouring lane (lane ^ 1) passes: a DPP move within each group of four lanes, no LDS.
__device__ __forceinline__ float swap_neighbours(float x) {
    int u = __float_as_int(x);
    return __int_as_float(__builtin_amdgcn_update_dpp(u, u, 0xB1, 0xf, 0xf, true));     // quad_perm [1, 0, 3, 2]
}
// x / (1 + exp(-x)) with the device's exponential and reciprocal instructions (each within an ulp; the result is
// rounded to bfloat16 right after).  For the epilogues that finish thousands of values per wave.
__device__ __forceinline__ float silu_fast_f32(float x) {
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x * -1.44269504088896341f));
}
// The tile loops' barrier: this wave's LDS reads and writes are done, then every wave of the block
// has arrived.  Unlike __syncthreads() it does not wait for loads from memory that are still in
// flight (the later tiles of a pipeline); the "memory" clobber keeps the compiler from moving
// memory accesses across it.
__device__ __forceinline__ void block_sync_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// All but the last N_ of this wave's vector memory operations have completed (they complete in order).
template <int N_>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N_ >= 0 && N_ < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt((N_ & 15) | (7 << 4) | (15 << 8) | ((N_ >> 4) << 14));
}

// Which tile of the output a block works on.  Blocks go to the eight XCDs in turn; here an XCD gets a stretch of the tiles
// that lie one after the other, eight rows of tiles at a time, column after column, so that the 32 blocks its units run at
// once are eight rows of four columns: each brings its rows of the weight into one L2, once, and shares them with seven
// others.  (Column after column over all XCDs, a grid of 224 columns gave an XCD 28 of them at once, each for one
// block: 2048 x 8192 times 57344 features 1773 -> 1473 us, 24576 x 4096 the same.)
// With rows shorter than 1024 the weight's bytes are few beside the results', and those are written faster as the grid counts its
// tiles (8192 x 128 times 28672 gated features 157 -> 145 us, 8192 x 256 added to 4096 100 -> 94; 8192 x 512
// times 8192 88 -> 83; with k of 128 and 16-bit results 1 % slower).
__device__ __forceinline__ void tile_of_block(int K, int& row, int& column) {
    row = blockIdx.y;
    column = blockIdx.x;
    if (K < 1024) return;
    int columns = gridDim.x, rows = gridDim.y, id = blockIdx.y * columns + blockIdx.x, share = columns * rows / 8;
    if (id < 8 * share) id = (id & 7) * share + (id >> 3);         // (what is left over when they do not divide by eight: as it comes)
    int band = id / (8 * columns), within = id - band * 8 * columns, high = min(8, rows - 8 * band);
    row = 8 * band + within % high;
    column = within / high;
}

// A wave's sums leave for 32-bit rows of `o`: FM x FN blocks of 16 tokens x 16 features, of which a lane holds four consecutive features of
// one token (token lane & 15, features 4 (lane >> 4) and on).  value(i, j) is a lane's f32x4, with HALF only the first two of it
// (gated pairs: an output for every two features).  A band of 16 tokens at a time goes through the wave's own part of LDS, `mine`
// (16 * (16 FN * 4 + 16) bytes, or half the features' of it), and leaves as whole lines, 16 bytes a lane where the rows allow that: stored from where
// they lie, 16 tokens' 64 bytes at a time, an instruction touches twice as many lines (2060 rows 16800 x 64 took 1.03 of the time, and
// rows of a number of features that four does not divide 1.3 of it).  Rows of the band lie 16 bytes more than their length apart, so
// that 16 tokens' pieces fall on different banks.  No waits: a wave's LDS accesses are carried out in the order it asks for them.
template <int FM, int FN, bool HALF, class Value>
__device__ __forceinline__ void bands_to_f32(unsigned char* mine, float* __restrict__ o, int ldc, int M, int N, int m_first, int n_first, bool add, Value&& value) {
    constexpr int COLS = HALF ? FN * 8 : FN * 16, ROW_BYTES = COLS * 4 + 16;
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & 63, token = lane & 15, g = lane >> 4;
    auto write = [&](auto ic) {
        constexpr int i = decltype(ic)::value;
        static_for<0, FN>([&](auto jc) {
            const f32x4 v = value(ic, jc);
            unsigned char* at = mine + token * ROW_BYTES + (decltype(jc)::value * (HALF ? 8 : 16) + g * (HALF ? 2 : 4)) * 4;
            if constexpr (HALF) *(f32x2*)at = f32x2{v[0], v[1]};
            else *(f32x4*)at = v;
        });
    };
    auto bands = [&](auto vec_of) {
        typedef decltype(vec_of) Vec;
        constexpr int W = sizeof(Vec) / 4, IN_ROW = COLS / W, PER = 16 * COLS / W / 64;
        static_assert(16 * COLS % (W * 64) == 0, "a band is the same number of pieces for every lane");
        auto place = [&](int i, int p, int& m, int& n) {
            const int at = p * 64 + lane;
            m = m_first + i * 16 + at / IN_ROW;
            n = n_first + at % IN_ROW * W;
        };
        Vec old[2][PER];
        auto ask = [&](auto ic) {
            constexpr int i = decltype(ic)::value;
#pragma unroll
            for (int p = 0; p < PER; ++p) {
                int m, n;
                place(i, p, m, n);
                old[i & 1][p] = add ? *(const Vec*)(o + (size_t)min(m, M - 1) * ldc + min(n, N - W)) : Vec{};
            }
        };
        ask(std::integral_constant<int, 0>{});
        write(std::integral_constant<int, 0>{});
        static_for<0, FM>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            Vec v[PER];
            asm volatile("" ::: "memory");
#pragma unroll
            for (int p = 0; p < PER; ++p) {
                const int at = p * 64 + lane;
                v[p] = *(const Vec*)(mine + at / IN_ROW * ROW_BYTES + at % IN_ROW * W * 4);
            }
            asm volatile("" ::: "memory");
            if constexpr (i + 1 < FM) {
                ask(std::integral_constant<int, i + 1>{});
                write(std::integral_constant<int, i + 1>{});
            }
#pragma unroll
            for (int p = 0; p < PER; ++p) {
                int m, n;
                place(i, p, m, n);
                if (m < M && n < N) *(Vec*)(o + (size_t)m * ldc + n) = old[i & 1][p] + v[p];
            }
            __builtin_amdgcn_sched_barrier(0);       // old values are asked for one band ahead, not all at once
        });
    };
    if (N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)o & 15) == 0) bands(f32x4{});      // (a lane's four features are in or out together)
    else if (N % 2 == 0 && ldc % 2 == 0 && ((uintptr_t)o & 7) == 0) bands(f32x2{});
    else bands(float{});
}

// Four consecutive features n .. n + 3 of one head of token m, as 32-bit sums, for the q/k/v epilogue: two rotation pairs
// (2i, 2i+1), rotated and rounded once; q to out, k and v into their places in the cache (never outside it).
template <class T>
__device__ __forceinline__ void store_qkv4(const QkvEpilogue& qe, void* __restrict__ out, int ldc, int m, int n, float (&v)[4]) {
    typedef T four __attribute__((ext_vector_type(4)));
    const int hd = qe.head_dim, head = n / hd, d = n % hd;
    const bool is_q = head < qe.n_heads, is_k = !is_q && head < qe.n_heads + qe.n_kv_heads;
    if (is_q || is_k) {
        const float pos = (float)qe.positions[m];
#pragma unroll
        for (int r = 0; r < 4; r += 2)
            if (d + r < qe.rotary_dim) {
                float sn, cs;
                sincosf(pos * qe.inv_freq[(d + r) >> 1], &sn, &cs);
                float a = v[r], b = v[r + 1];
                v[r] = a * cs - b * sn;
                v[r + 1] = a * sn + b * cs;
            }
    }
    four o4;
#pragma unroll
    for (int r = 0; r < 4; ++r) o4[r] = from_f32<T>(v[r]);
    if (is_q) {
        *(four*)((T*)out + (size_t)m * ldc + n) = o4;
    } else if (qe.write_kv) {
        const int slot = qe.slot_map[m];
        if (slot < 0 || slot >= qe.num_pages * qe.page_size) return;
        const int page = slot / qe.page_size, off = slot % qe.page_size, kvh = head - qe.n_heads - (is_k ? 0 : qe.n_kv_heads);
        if (is_k) {
            *(four*)((T*)qe.k_cache + k_cache_index(page, kvh, off, d, qe.n_kv_heads, qe.page_size, hd)) = o4;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                ((T*)qe.v_cache)[v_cache_index(page, kvh, off, d + r, qe.n_kv_heads, qe.page_size, hd)] = o4[r];
        }
    }
}
