// Products of up to 16 rows (decoding), in 32-bit up to 32 (some of one and two rows go to gemm_rows_kernel), bfloat16 and 32-bit, on the matrix cores with 32-bit sums.
//
// What bounds them: the weight's bytes, each read once, how many of them are on their way at a time, and the address unit in
// front of the vector cache, which takes a line a clock.  A block owns 8 NG output features; its NW waves take the k-blocks
// (128 bytes of a row: 64 bfloat16 or 32 32-bit numbers) in turn and add their sums through LDS in wave order.  Every wave has
// a ring of R k-blocks in LDS to itself: loads straight into LDS bring whole lines, eight rows of 128 bytes to an
// instruction (an operand read straight from memory is 16 rows to 16 lanes, 64 lines to an instruction; in a block of 8 features
// with 8 tokens that was 33,000 clocks of 2048 x 8192 32-bit numbers' 48,000), no barrier stands between them, and the
// next ones are on their way while this one is multiplied.  Chunk c of row r lies in slot c ^ (r & 7) of its row: eight lanes' reads
// hit eight bank groups.
//
// v_mfma_f32_16x16x32_bf16 and v_mfma_f32_16x16x4_f32 multiply 16 rows of the weight (operand A) by 16 tokens (operand B).
//   Up to 8 tokens (FOLD) half of that would be work for rows that are not there, so the operands are folded: their 16 rows are
//   8 features, and 8 tokens, in each of the two halves of a k-block.  One MFMA (four in 32-bit) contracts the whole
//   k-block, and of its 16 x 16 results the two 8 x 8 blocks on the diagonal are the halves' sums.
//   9 to 16 tokens: an operand is 16 features, or 16 tokens, of one half of a k-block, and the two halves have sums of their own;
//   17 to 32: the same with TT = 2 tiles of tokens.
// Either way an output is the sum of each wave's (first halves' sum + second halves' sum), in bfloat16 in wave order: its
// bits depend on K and on the weight's shape, which choose NW and where a block's walk along k begins, never on M.
// (In 32-bit the waves' sums are added pairwise, and bits differ by rounding between up to 2, up to 8, up to 16 and more rows.)
// Measured, 16 features an operand and operands from memory -> as here (MI355X, weights from memory, us): bfloat16 at 1 row
// 2048 x 8192 12.3 -> 8.6, 2048 x 2048 5.7 -> 4.3, 128256 x 2048 90 -> 83 (6.3 TB/s); at 8 rows 4096 x 4096 11.4 -> 8.6, 4096 x 14336
// 28.5 -> 23.2, 28672 x 4096 44.2 -> 42.0; at 16 rows 4096 x 4096 13.3 -> 8.5, 4096 x 14336 35 -> 24.7, 10240 x 8192 49.5 -> 34.6;
// 32-bit at 8 rows 2048 x 8192 26.1 -> 15.5, 2048 x 32768 88 -> 52, 16384 x 2048 28.8 -> 25.9, 128256 x 2048 187 -> 174.
#include "gemm_tile.h"
#include "recurrent.h"

template <class T> struct Few;
template <> struct Few<bf16> { typedef bf16x8 Piece; typedef bf16x4 Four; };
template <> struct Few<float> { typedef f32x4 Piece; typedef f32x4 Four; };

// The sums of a tile: a 32-bit piece is four MFMAs, whose products go to SUMS sums of their own (eight: those of every other k-block
// to the second four), added pairwise at the end: a quarter or an eighth of the products one after the other in a sum, and an error
// against 64 bits to match.
template <class T, int SUMS>
struct FewSums {
    f32x4 s[SUMS];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int i = 0; i < SUMS; ++i) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    template <int HALF>
    __device__ __forceinline__ void add(const typename Few<T>::Piece& w, const typename Few<T>::Piece& x) {
        if constexpr (sizeof(T) == 2) s[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, s[0], 0, 0, 0);
        else {
#pragma unroll
            for (int j = 0; j < 4; ++j) s[(4 * HALF + j) % SUMS] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], s[(4 * HALF + j) % SUMS], 0, 0, 0);
        }
    }
    __device__ __forceinline__ f32x4 total() const {
        if constexpr (SUMS == 8) return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
        else if constexpr (SUMS == 4) return (s[0] + s[1]) + (s[2] + s[3]);
        else if constexpr (SUMS == 2) return s[0] + s[1];
        else return s[0];
    }
};
// In lanes 0..7 and 16..23: the sum with the lane 40 further on (the other half of the k-blocks, see above).
__device__ __forceinline__ float with_other_half(float x) {
    unsigned u = __float_as_uint(x);
    auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);       // [1]: in the low lanes the values of the high ones
    int far = (int)sw[1];
    return x + __int_as_float(__builtin_amdgcn_update_dpp(far, far, 0x128, 0xf, 0xf, true));     // row_ror:8
}

// What a call brings beyond its operands, a kernel for each kind: an argument's trip from memory in front of the first load
// costs a product of few microseconds a tenth of its time (1 row of 2048 x 2048 bfloat16, with all of them 5.1 us, with none 4.45).
struct FewPlain {};
struct FewScaled { RowScale scale; };
struct FewNext { RowScale scale; NextNorm next; };
struct FewQkv { RowScale scale; QkvEpilogue qkv; };
// Products of a recurrent mixer in a step where every request brings one token: what the mixer does with the sums, channel by channel
// and request by request, is done where they are finished (rows: requests; `slots` their state's rows; states 32-bit).  A kernel of its
// own for it took 4.8 us for a few KB, three trips to memory one after the other, and 1.3 more between two kernels; here the
// trips for the state run beside the weight's.  (4 requests, product and kernel -> here, us: convolution, 8192 x 2048, 8.2 + 4.8 ->
// 8.4; minGRU, 6144 x 2048, 7.0 + 4.7 -> 8.0; scan, 4096 x 128, 4.7 + 4.9 -> 5.5.)
//   FewConv: features below C are inputs of the causal convolution of four taps (recurrent.hip): silu of it goes to x, the state's three
//     rows move on; the features above go to `out` in 32-bit.
//   FewGru: the weight's rows are (gate | candidate | output gate), a third each; a block takes eight channels of all three
//     (an eight of rows each), advances the state and writes the gated one to `out`.
//   FewScan: the sums are the step sizes of a selective scan of 16 states: the state's step, the output to `out`.  A thread for each
//     request and channel of the block.
struct FewConv { const float* taps; const float* bias; float* state; long state_stride; const int* slots; bf16* x; int ldx, C; };
struct FewGru { const float* bias_z; const float* bias_c; float* state; long state_stride; const int* slots; };
struct FewScan {
    const float* dt_bias; const float* A; const float* D; const float* gate; float* state; long state_stride; const int* slots;
    const bf16* x; const bf16* b; const bf16* c;       // b, c: row 0's 16 of either, rows ldbc apart
    int ld_gate, ldx, ldbc;
};
constexpr int SCAN_STATES = 16;
template <class Extra> constexpr bool few_scaled = std::is_same<Extra, FewScaled>::value || std::is_same<Extra, FewNext>::value || std::is_same<Extra, FewQkv>::value;
template <class T, bool FOLD, int NG, int NW, int R, int ROT, int SUMS, int TT, class Extra>
__global__ __launch_bounds__(NW * 64) void gemm_few_kernel(const T* __restrict__ A, const T* __restrict__ W, void* __restrict__ out, int lda,
                                                           int ldc, int M, int N, int K, int epi, unsigned inv_full, Extra extra) {
    constexpr bool NEXT = std::is_same<Extra, FewNext>::value, QKV = std::is_same<Extra, FewQkv>::value;
    constexpr bool CONV = std::is_same<Extra, FewConv>::value, GRU = std::is_same<Extra, FewGru>::value, SCAN = std::is_same<Extra, FewScan>::value;
    static_assert(!GRU || NG == 3, "an eight of rows of each of the three projections");
    static_assert(!SCAN || (NG == 2 && NW == 4), "a thread for each of 16 requests and 16 channels");
    RowScale rs{};
    NextNorm nn{};
    QkvEpilogue qe{};
    if constexpr (few_scaled<Extra>) rs = extra.scale;
    if constexpr (NEXT) nn = extra.next;
    if constexpr (QKV) qe = extra.qkv;
    typedef typename Few<T>::Piece Piece;
    typedef typename Few<T>::Four Four;
    constexpr int PER = 16 / (int)sizeof(T), KB = 8 * PER;         // numbers in a lane's piece, in a k-block
    constexpr int TILES = (NG + 1) / 2;                            // tiles of 16 features (the last one half, where NG is odd)
    constexpr int TOK = FOLD ? 8 : 16;
    constexpr int WL = FOLD ? NG : TILES * 2, XL = FOLD ? 1 : 2 * TT;   // a lane's pieces of a k-block: weight, tokens (TT tiles of them)
    static_assert(TT == 1 || !FOLD, "folded operands are of eight tokens");
    constexpr int LOADS = NG + XL, BLOCK = LOADS * 1024;           // a k-block in LDS: eight rows of 128 bytes to a load
    static_assert((R - 2) * LOADS < 64 && R >= 2, "vmcnt counts to 63");
    extern __shared__ __attribute__((aligned(1024))) unsigned char few_smem[];
    f32x4* red = (f32x4*)(few_smem + NW * R * BLOCK);              // [NW][TT][NG][2: four features each][TOK]
    float* scale_red = (float*)(red + NW * TT * NG * 2 * TOK);     // [NW][16]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * NG * 8;
    auto weight_row = [&](int group, int r) { return min(GRU ? group * (N / 3) + (int)blockIdx.x * 8 + r : n0 + group * 8 + r, N - 1); };   // row r of a block's eight
    // the rows that this lane's part of a load is of, at the chunk that belongs in the lane's slot
    const T* src[LOADS];
    {
        const int lrow = lane >> 3, chunk = ((lane & 7) ^ lrow) * PER;
#pragma unroll
        for (int i = 0; i < NG; ++i) src[i] = W + (size_t)weight_row(i, lrow) * K + chunk;
#pragma unroll
        for (int i = 0; i < XL; ++i) src[NG + i] = A + (size_t)min(i * 8 + lrow, M - 1) * lda + chunk;
    }
    FewSums<T, SUMS> acc[TT][WL];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int i = 0; i < WL; ++i) acc[tt][i].clear();

    // A norm left to this product (RowScale): its partial sums of squares are shared out over the waves and asked for before
    // the weights, so that their trip to memory (they were written on other XCDs) costs nothing beside the weights'.
    // (Asked for after the walk along k it was a trip in front of every result: 0.9 us of the product.)
    constexpr int AHEAD = 4;
    const bool scaled = TT == 1 && few_scaled<Extra> && rs.sumsq != nullptr, by_four = rs.nparts % 16 == 0 && ((uintptr_t)rs.sumsq & 15) == 0;
    const float* sp = rs.sumsq + (size_t)min(row, M - 1) * rs.nparts;
    f32x4 part[AHEAD];
    if (scaled && by_four) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            int at = 16 * (wave + NW * i) + 4 * g;
            part[i] = at < rs.nparts ? *(const f32x4*)(sp + at) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // out += sum: the old values of the tile this wave will finish, and the next norm's weight for them, likewise
    float old[4] = {0.0f, 0.0f, 0.0f, 0.0f}, next_w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const bool old_ahead = !QKV && epi == LLMRS_EPI_ACCUM_F32 && wave < TILES * TT;
    const int own = wave % TILES, own_m = wave / TILES * 16 + row;          // that tile, and this lane's token of it
    if (old_ahead && own_m < M) {
        int n = n0 + own * 16 + 4 * g;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (n + r < N && 4 * g < 8 * NG - 16 * own) {
                old[r] = ((const float*)out)[(size_t)own_m * ldc + n + r];
                if (NEXT) next_w[r] = nn.weight[n + r];
            }
    }

    // a recurrent mixer's step: everything that it reads beside the sums
    f32x4 was[3] = {}, tap[4] = {}, lane_bias[2] = {};
    float* state_at = nullptr;
    if constexpr (CONV) {
        const int n = n0 + wave * 16 + 4 * g;
        if (wave < TILES && 2 * wave + (g >> 1) < NG && row < M && n < extra.C) {
            state_at = extra.state + (size_t)extra.slots[row] * extra.state_stride + n;
            lane_bias[0] = extra.bias ? *(const f32x4*)(extra.bias + n) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < 4; ++r) tap[r] = *(const f32x4*)(extra.taps + (size_t)(n + r) * 4);
#pragma unroll
            for (int j = 0; j < 3; ++j) was[j] = *(const f32x4*)(state_at + (size_t)j * extra.C);
        }
    }
    if constexpr (GRU) {
        const int c = blockIdx.x * 8 + 4 * g;
        if (wave == 0 && g < 2 && row < M) {
            state_at = extra.state + (size_t)extra.slots[row] * extra.state_stride + c;
            lane_bias[0] = extra.bias_z ? *(const f32x4*)(extra.bias_z + c) : f32x4{0.f, 0.f, 0.f, 0.f};
            lane_bias[1] = extra.bias_c ? *(const f32x4*)(extra.bias_c + c) : f32x4{0.f, 0.f, 0.f, 0.f};
            was[0] = *(const f32x4*)state_at;
        }
    }
    float S[SCAN ? SCAN_STATES : 1], Ac[SCAN ? SCAN_STATES : 1], xv = 0.0f, gv = 0.0f, Dc = 0.0f, dt0 = 0.0f;
    bf16x8 Bn[2], Cn[2];
    const int sm = threadIdx.x >> 4, sf = threadIdx.x & 15;        // SCAN: this thread's request, and its channel of the block's
    if constexpr (SCAN) {
        const int c = n0 + sf;
        if (sm < M) {
            state_at = extra.state + (size_t)extra.slots[sm] * extra.state_stride + c;          // state n of the channel: state_at[n N]
#pragma unroll
            for (int n = 0; n < SCAN_STATES; ++n) Ac[n] = extra.A[(size_t)n * N + c];
            Dc = extra.D[c];
            dt0 = extra.dt_bias ? extra.dt_bias[c] : 0.0f;
            gv = extra.gate[(size_t)sm * extra.ld_gate + c];
            xv = to_f32(extra.x[(size_t)sm * extra.ldx + c]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                Bn[h] = *(const bf16x8*)(extra.b + (size_t)sm * extra.ldbc + 8 * h);
                Cn[h] = *(const bf16x8*)(extra.c + (size_t)sm * extra.ldbc + 8 * h);
            }
#pragma unroll
            for (int n = 0; n < SCAN_STATES; ++n) S[n] = state_at[(size_t)n * N];
        }
    }

    const int full = (unsigned)K / KB;
    // A block's walk along k begins at a k-block of its own and wraps round: rows are a multiple of the memory channels'
    // interleave apart, so blocks in step would all ask the same few channels at once.  The start depends on the group of ROT
    // features alone that the block's lie in, not on how many it takes: `step` times the group's number, modulo the k-blocks
    // (by a product with `inv_full`, 2^32 / full rounded up: exact for what fits in 16 bits, and any start will do).
    int rot = 0;
    if constexpr (ROT > 0) {
        // (Of groups of 112 features, rows that are no multiple of 16 KB want neighbours a k-block apart: with 1 in place of 37, up to 8 rows of 18944 to
        // 57344 x 4096 in bfloat16 and x 2048 in 32-bit take 0.86-0.91 of the time, 37888 x 2048 or 28672 x 3072 the same; rows of 16 KB 1.08-1.16
        // of it.  Smaller groups of rows of 16 KB: 4096 x 8192 in bfloat16 1.11, in 32-bit 1.24; of 8 KB 0.97-1.02.)
        const unsigned step = ROT == 112 && (unsigned)K % (16384 / sizeof(T)) != 0 ? 1u : 37u;
        unsigned start = (unsigned)n0 / ROT * step & 0xffffu;
        rot = full > 1 ? (int)(start - __umulhi(start, inv_full) * (unsigned)full) : 0;
    }
    // This wave's k-blocks, the wave + NW i'th of the walk, through a ring of R places of its own: R - 1 of them on their way.
    // Loads complete in order, so a k-block has landed when all but the loads behind its own have; the place that the next
    // one goes into was read for the products before.
    unsigned char* ring = few_smem + wave * (R * BLOCK);
    const int mine = (full - wave + NW - 1) / NW;
    int at = wave + rot, put = 0;                                  // of the next k-block asked for: its place in the row, and in the ring
    auto ask = [&] {
        const size_t k = (size_t)(at >= full ? at - full : at) * KB;
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + k),
                                             (__attribute__((address_space(3))) void*)(ring + __builtin_amdgcn_readfirstlane(put * BLOCK + i * 1024)), 16, 0, 0);
        at += NW;
        put = put + 1 == R ? 0 : put + 1;
    };
    auto products = [&](auto half, const Piece (&w)[WL], const Piece (&x)[XL]) {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int i = 0; i < WL; ++i) acc[tt][i].template add<decltype(half)::value>(w[i], x[FOLD ? 0 : 2 * tt + (i & 1)]);
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
#pragma unroll
    for (int i = 0; i < R - 1; ++i)
        if (i < mine) ask();
    const int f = row & 7;
    const int off0 = f * 128 + (((FOLD ? (row >> 3) * 4 + g : g) ^ f) * 16), off1 = f * 128 + (((4 + g) ^ f) * 16);      // a lane's pieces of eight rows
    for (int i = 0, get = 0; i < mine; ++i, get = get + 1 == R ? 0 : get + 1) {
        if (i + R - 1 <= mine) wait_vmcnt<(R - 2) * LOADS>(); else wait_vmcnt<0>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // (the place about to be filled has been read)
        if (i + R - 1 < mine) ask();
        const unsigned char* b = ring + get * BLOCK;
        Piece w[WL], x[XL];
        if constexpr (FOLD) {
            x[0] = *(const Piece*)(b + NG * 1024 + off0);
#pragma unroll
            for (int t = 0; t < NG; ++t) w[t] = *(const Piece*)(b + t * 1024 + off0);
        } else {
            const int half = (row >> 3) * 1024;
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                x[2 * tt] = *(const Piece*)(b + (NG + 2 * tt) * 1024 + half + off0);
                x[2 * tt + 1] = *(const Piece*)(b + (NG + 2 * tt) * 1024 + half + off1);
            }
            // (with an odd number of groups the last tile's other half reads the tokens' rows: its sums are not used)
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                w[2 * t] = *(const Piece*)(b + t * 2048 + half + off0);
                w[2 * t + 1] = *(const Piece*)(b + t * 2048 + half + off1);
            }
        }
        if (SUMS == 8 && (i & 1)) products(odd, w, x); else products(even, w, x);
    }
    if (K % KB != 0 && wave == full % NW) {      // the k-block that K cuts, straight from memory
        const int k = full * KB, first = (FOLD ? (row >> 3) * 4 + g : g) * PER;
        Piece w[WL], x[XL];
#pragma unroll
        for (int i = 0; i < WL; ++i) {
            const int n = FOLD ? weight_row(i, f) : weight_row(i / 2 * 2 + (row >> 3), f), from = k + first + (FOLD ? 0 : (i % 2) * (KB / 2));
            w[i] = from < K ? *(const Piece*)(W + (size_t)n * K + from) : Piece{};
        }
#pragma unroll
        for (int i = 0; i < XL; ++i) {
            const int from = k + first + (i & 1) * (KB / 2);
            x[i] = from < K ? *(const Piece*)(A + (size_t)min(FOLD ? f : i / 2 * 16 + row, M - 1) * lda + from) : Piece{};
        }
        products(even, w, x);
    }
    if (scaled) {
        float ss = 0.0f;
        if (by_four) {
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) ss += (part[i][0] + part[i][1]) + (part[i][2] + part[i][3]);
            for (int at = 16 * (wave + NW * AHEAD) + 4 * g; at < rs.nparts; at += 16 * NW) {
                f32x4 p = *(const f32x4*)(sp + at);
                ss += (p[0] + p[1]) + (p[2] + p[3]);
            }
        } else {
            for (int at = 4 * wave + g; at < rs.nparts; at += 4 * NW) ss += sp[at];
        }
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        if (g == 0) scale_red[wave * 16 + row] = ss;
    }
    if constexpr (FOLD) {
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            f32x4 s = acc[0][i].total();
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = with_other_half(s[r]);
            if (row < 8 && g < 2) red[((wave * NG + i) * 2 + g) * TOK + row] = s;
        }
    } else {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                if (2 * t + (g >> 1) < NG) red[(((wave * TT + tt) * NG + 2 * t) * 2 + g) * TOK + row] = acc[tt][2 * t].total() + acc[tt][2 * t + 1].total();
    }
    __syncthreads();
    if constexpr (GRU) {
        if (wave > 0 || g > 1 || row >= M) return;
        f32x4 v[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < NW; ++w) v[i] += red[((w * NG + i) * 2 + g) * TOK + row];
        }
        f32x4 s;
        Four y;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = mingru_state(was[0][r], sigmoid_f32(v[0][r] + lane_bias[0][r]), v[1][r] + lane_bias[1][r]);
            y[r] = from_f32<T>(s[r] * silu_f32(v[2][r]));
        }
        *(f32x4*)state_at = s;
        *(Four*)((T*)out + (size_t)row * ldc + blockIdx.x * 8 + 4 * g) = y;
        return;
    }
    if constexpr (SCAN) {
        if (sm >= M) return;
        float vdt = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) vdt += ((const float*)red)[(((w * NG + (sf >> 3)) * 2 + (sf >> 2 & 1)) * TOK + sm) * 4 + (sf & 3)];
        const float step = softplus_f32(vdt + dt0), sx = step * xv;
        float y = 0.0f;
#pragma unroll
        for (int n = 0; n < SCAN_STATES; ++n) {
            S[n] = fmaf(__builtin_amdgcn_exp2f(step * (Ac[n] * LOG2_E)), S[n], sx * (float)Bn[n / 8][n % 8]);
            y = fmaf(S[n], (float)Cn[n / 8][n % 8], y);
            state_at[(size_t)n * N] = S[n];
        }
        y = fmaf(Dc, xv, y);
        ((T*)out)[(size_t)sm * ldc + n0 + sf] = from_f32<T>(y * silu_f32(gv));
        return;
    }
    // the tiles are shared out over the waves: lane l finishes token l % 16 and features 4 (l / 16) + r
    if (wave >= TILES * TT || (TT == 1 && row >= M)) return;
    float inv = 1.0f;
    if (scaled) {
        float total = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) total += scale_red[w * 16 + row];
        inv = 1.0f / sqrtf(total / (float)K + rs.eps);
    }
    for (int which = wave; which < TILES * TT; which += NW) {
        const int tile = which % TILES, tt = which / TILES, m = tt * 16 + row;
        if (m >= M || 2 * tile + (g >> 1) >= NG) continue;         // (the half of the last tile is the next block's)
        f32x4 of[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) of[w] = red[(((w * TT + tt) * NG + 2 * tile) * 2 + g) * TOK + row];
        f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (sizeof(T) == 2) {
#pragma unroll
            for (int w = 0; w < NW; ++w) s += of[w];
        } else {
            // pairwise: up to 8 rows of K = 2048 are 1.22e-7 off the 64-bit result, in wave order 1.26e-7
#pragma unroll
            for (int step = 1; step < NW; step *= 2)
#pragma unroll
                for (int w = 0; w < NW; w += 2 * step) of[w] += of[w + step];
            s = of[0];
        }
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = s[r] * inv;
        const int n = n0 + tile * 16 + 4 * g;
        if constexpr (CONV) {
            static_assert(TILES <= NW, "a wave finishes the one tile whose state it has asked for");
            if (n >= N) continue;
            if (n >= extra.C) {
                *(f32x4*)((float*)out + (size_t)m * ldc + n) = f32x4{v[0], v[1], v[2], v[3]};
                continue;
            }
            Four y;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float a = lane_bias[0][r];
#pragma unroll
                for (int j = 0; j < 3; ++j) a = fmaf(tap[r][j], was[j][r], a);
                y[r] = from_f32<T>(silu_f32(fmaf(tap[r][3], v[r], a)));
            }
            *(f32x4*)state_at = was[1];
            *(f32x4*)(state_at + extra.C) = was[2];
            *(f32x4*)(state_at + (size_t)2 * extra.C) = f32x4{v[0], v[1], v[2], v[3]};
            *(Four*)((T*)extra.x + (size_t)m * extra.ldx + n) = y;
            continue;
        }
        if (!NEXT && !QKV && epi_gated(epi)) {
#pragma unroll
            for (int r = 0; r < 4; r += 2)
                if (n + r + 1 < N) ((T*)out)[(size_t)m * ldc + (n + r) / 2] = from_f32<T>(gated_act(epi, v[r], v[r + 1]));
        } else if (QKV) {
            if (n < N) store_qkv4<T>(qe, out, ldc, m, n, v);
        } else if (old_ahead && which == wave) {
            float ss = 0.0f;
            Four y4;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float nv = 0.0f;
                if (n + r < N) {
                    nv = old[r] + v[r];
                    ((float*)out)[(size_t)m * ldc + n + r] = nv;
                    ss = fmaf(nv, nv, ss);
                    nv *= next_w[r];
                }
                y4[r] = from_f32<T>(nv);
            }
            if (NEXT) {
                // for the norm that follows (NextNorm).  The row's lanes hold four features each; they are all here: a row is
                // in the batch for all of them or for none.
                T* y = (T*)nn.y + (size_t)m * nn.ldy + n;
                if (n + 3 < N) *(Four*)y = y4;
                else
                    for (int r = 0; r < 4; ++r)
                        if (n + r < N) y[r] = y4[r];
                ss += __shfl_xor(ss, 16, 64);
                if constexpr (NG == 1) {
                    if (g == 0) nn.sumsq[(size_t)m * ((N + 7) / 8) + n0 / 8] = ss;        // a part is the block's 8 features
                } else {
                    ss += __shfl_xor(ss, 32, 64);
                    if (g == 0) nn.sumsq[(size_t)m * ((N + 15) / 16) + (n0 / 16 + tile)] = ss;
                }
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) epilogue_store<T>(epi, out, ldc, m, n + r, v[r]);
        }
    }
}

struct FewCall {
    hipStream_t stream;
    const void* A;
    int lda;
    const void* W;
    void* out;
    int ldc, M, N, K, epi;
    QkvEpilogue qkv;
    RowScale scale;
    NextNorm next;
};
template <class T, bool FOLD, int NG, int NW, int R, int ROT, int SUMS = 1, int TT = 1, class Launch>
static void with_few_launcher(const FewCall& c, Launch choose) {
    static_assert(ROT % (NG * 8) == 0, "a block's features lie in one group");
    const unsigned full = c.K * sizeof(T) / 128, inv_full = full > 1 ? (unsigned)(((1ull << 32) + full - 1) / full) : 0;
    constexpr size_t bytes = (size_t)NW * R * (NG + (FOLD ? 1 : 2 * TT)) * 1024 + (size_t)NW * TT * NG * 2 * (FOLD ? 8 : 16) * 16 + NW * 16 * sizeof(float);
    static_assert(bytes <= 160 * 1024, "the rings and the waves' sums must fit in a unit's LDS");
    auto launch = [&](auto extra) {
        static bool configured = false;
        if (!configured) {
            (void)hipFuncSetAttribute((const void*)gemm_few_kernel<T, FOLD, NG, NW, R, ROT, SUMS, TT, decltype(extra)>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
            configured = true;
        }
        gemm_few_kernel<T, FOLD, NG, NW, R, ROT, SUMS, TT><<<ceil_div(c.N, NG * 8), NW * 64, bytes, c.stream>>>(
            (const T*)c.A, (const T*)c.W, c.out, c.lda, c.ldc, c.M, c.N, c.K, c.epi, inv_full, extra);
    };
    choose(launch);
}
template <class T, bool FOLD, int NG, int NW, int R, int ROT, int SUMS = 1, int TT = 1>
static void launch_few(const FewCall& c) {
    with_few_launcher<T, FOLD, NG, NW, R, ROT, SUMS, TT>(c, [&](auto launch) {
        if constexpr (TT > 1) launch(FewPlain{});             // (more than 16 rows: no norm is left to them, and no rotation)
        else if (c.epi == LLMRS_EPI_QKV) launch(FewQkv{c.scale, c.qkv});
        else if (c.next.y != nullptr) launch(FewNext{c.scale, c.next});
        else if (c.scale.sumsq != nullptr) launch(FewScaled{c.scale});
        else launch(FewPlain{});
    });
}
// Whether blocks of 24 features (a tile and a half) share a weight of N features out over the device's units more
// evenly, by a tenth of a round or more, than blocks of `whole` features (16 or 32) do.
bool llmrs_half_tile_blocks(int N, int whole, int cus) {
    auto even = [&](int b) { return (double)b / ((double)ceil_div(b, cus) * cus); };
    return N % 8 == 0 && even(ceil_div(N, 24)) > even(ceil_div(N, whole)) + 0.1;
}
// A narrow weight with long rows (16-feature blocks would leave half of the compute units without one): blocks of 8 features.
static bool half_blocks_for_narrow(int N, int K) {
    return N < 16384 && K >= 2048 && N % 8 == 0 && ceil_div(N, 16) * 2 <= llmrs_compute_units();
}
// Whether a wide weight's blocks fill the device's units more evenly by 7 or by 4 tiles of 16 features
// (28672 features are 256 blocks of 7 tiles).
static int wide_tiles(int N, int cus) {
    auto evenness = [&](int nt) { int b = ceil_div(N, 16 * nt); return (double)b / ((double)ceil_div(b, cus) * cus); };
    return evenness(7) >= evenness(4) ? 7 : 4;
}
extern "C" int llmrs_gemm_defers_norm(int M, int N, int K) { return M >= 1 && M <= 16 && N >= 1 && K % 8 == 0; }
// (one row on the widest weights: the norm's kernel and gemm_rows_kernel together are faster, 128256 x 2048 175.6 against 180.0 us; 2 rows 182 and 179.5)
extern "C" int llmrs_gemm_f32_defers_norm(int M, int N, int K) { return M >= 1 && M <= 16 && N >= 1 && K % 32 == 0 && !(M == 1 && N >= 65536); }
extern "C" int llmrs_gemm_leaves_norm(int N) { return N < 16384 && N % 4 == 0; }
extern "C" int llmrs_qkv_by_fours(int head_dim, int rotary_dim) { return head_dim % 4 == 0 && rotary_dim % 4 == 0; }
extern "C" int llmrs_gemm_next_parts(int M, int N, int K) {
    return M <= 16 && half_blocks_for_narrow(N, K) ? ceil_div(N, 8) : ceil_div(N, 16);
}

// Up to 8 rows: blocks of 8 NG features, rings of R k-blocks, in 32-bit four sums a tile; 9 to 16 rows: of 8 NG16, R16, one sum: the
// error of the 32-bit products against 64 bits is then no larger than it was with one sum for whole k-blocks (K = 2048: 1.25e-7
// up to 8 rows, 2.1e-7 from 9 on, against 2.9e-7).
template <class T, int NW, int ROT, int NG, int R, int NG16, int R16>
static void launch_few_by_rows(const FewCall& c) {
    if (c.M <= 8) launch_few<T, true, NG, NW, R, ROT, sizeof(T) == 4 ? 4 : 1>(c);
    else launch_few<T, false, NG16, NW, R16, ROT>(c);
}
// Waves per block and the walk's start come from the weight's shape alone (see above).  With fewer features a block, more blocks
// ask at once but each reads the tokens' rows again.  Rings of three k-blocks do nearly as well as any: what is on its way
// is then some 32 KB of the weight a unit.
// 17 to 32 rows in 32-bit: two tiles of tokens for every piece of the weight, which is read once.  (us at 32 rows against
// gemm_f32_skinny_kernel, whose operands come straight from memory and touch eight times the cache lines: 2048 x 2048 15.1 -> 9.4,
// 2048 x 8192 46.2 -> 27.7, 3072 x 2048 14.4 -> 10.7, 16384 x 2048 33.4 -> 29.9, 28672 x 4096 148 -> 90, 128256 x 2048 312 -> 206;
// 8192 x 28672 239 -> 191.)  The shares of k are half as long and two sums run beside each other: the error against 64 bits is smaller.
// The widest weights want many features a block, as each block reads the tokens' rows again (128256 x 2048: 64 features 206, 32
// 230-245, 16 285); the narrow ones enough blocks (3072 x 2048: 16 features 10.7, 8 16.9).
static void few_rows_two_tiles(const FewCall& c) {
    if (c.N >= 16384) launch_few<float, false, 8, 4, 2, 64, 1, 2>(c);
    else if (c.K < 2048) launch_few<float, false, 2, 4, 2, 0, 1, 2>(c);
    else if (c.N >= 8192) launch_few<float, false, 4, 4, 3, 64, 1, 2>(c);
    else if (half_blocks_for_narrow(c.N, c.K)) launch_few<float, false, 1, 8, 2, 64, 1, 2>(c);
    else launch_few<float, false, 2, 8, 2, 0, 1, 2>(c);
}
// One and two rows in 32-bit: eight waves and eight sums a tile whatever the shape.  gemm_rows_kernel, which takes such products too (see
// llmrs_gemm), adds up few numbers one after the other, and the error here is to be no larger: K = 1024 0.9e-7 against 1.0e-7, 2048 1.02
// and 1.23, 4096 1.27 and 1.59 (with four waves and four sums 1.2, 1.57 and 2.1); with a norm left to the product, against the norm's kernel and
// gemm_rows_kernel, 320 1.0e-7 both, 2048 1.18 and 1.33.
static void few_rows_one_or_two(const FewCall& c) {
    const int N = c.N, K = c.K, cus = llmrs_compute_units();
    if (N >= 16384) launch_few<float, true, 2, 8, 3, 64, 8>(c);
    else if (K >= 16384 && N >= 8192) launch_few<float, true, 4, 8, 2, 64, 8>(c);
    else if (half_blocks_for_narrow(N, K)) launch_few<float, true, 1, 8, 5, 64, 8>(c);
    else if (c.next.y == nullptr && K >= 2048 && llmrs_half_tile_blocks(N, 16, cus)) launch_few<float, true, 3, 8, 3, 96, 8>(c);
    else launch_few<float, true, 2, 8, 3, 64, 8>(c);
}
template <class T>
static void few_rows(const FewCall& c) {
    const int N = c.N, K = c.K, cus = llmrs_compute_units();
    if (sizeof(T) == 4 && c.M > 16) { few_rows_two_tiles(c); return; }
    if (sizeof(T) == 4 && c.M <= 2) { few_rows_one_or_two(c); return; }
    const int kblocks = ceil_div(K * (int)sizeof(T), 128);
    // Short rows, and more than two blocks of 16 features a unit: what fills the time is the other blocks, not a deep ring, which a wave has not
    // the k-blocks to fill and which keeps blocks off the unit (us, rings of three to five in blocks of 16 to 64 features -> as here: 32-bit at 8
    // rows 65536 x 256 22.9 -> 15.9, 100000 x 128 27 -> 14.6, 13824 x 256 6.7 -> 5.6, at 16 rows 32000 x 256 12.8 -> 9.6; bfloat16 at 8 rows
    // 65536 x 512 20 -> 14.8, at 16 50304 x 256 13 -> 8.9).  From 32 k-blocks on the rings gain (bfloat16 at 1 row 32000 x 2560 30.7, as here 31.3).
    if (kblocks <= 16 && ceil_div(N, 16) > 2 * cus) {
        // (the shortest of them, many features: two waves a block.  32-bit 100000 x 128 at 16 rows 17.6 with four, 15.7 with two; bfloat16 65536 x 512
        // at 12 rows 16.1 and 15.6, 32000 x 256 6.6 and 5.8; 13824 x 128 at 8 rows 4.4 and 5.1)
        if (kblocks <= (sizeof(T) == 2 ? 8 : 4) && N >= 24576) launch_few_by_rows<T, 2, 64, 4, 2, 4, 2>(c);
        else launch_few_by_rows<T, 4, 0, 2, 2, 2, 2>(c);
    }
    else if (N >= 16384) {
        // (28672 x 4096 bfloat16 at 8 rows: blocks of 16 features 42.0 us, of 56 43.7, of 112 47; at 16 rows of 56 41.8, of 112 42.4)
        if (wide_tiles(N, cus) == 7) launch_few_by_rows<T, 4, 112, 2, 4, 7, 3>(c);
        // (at 16 rows 16384 x 2048: blocks of 64 features 14.5, of 16 15.1; in 32-bit, where a k-block is more MFMAs, of 32 25.8, of 16 27.2, 32000 x 2560
        // 62.5 and 70.5, 128256 x 2048 181 and 200)
        else if (c.M > 8) { if (sizeof(T) == 2) launch_few<T, false, 8, 4, 3, 64>(c); else launch_few<T, false, 4, 4, 2, 64>(c); }
        // (deeper rings let fewer blocks share a unit: 16384 x 2048 at 8 rows 14.3 with three, 14.9 with five; 128256 x 2048 93.2 and 90.9)
        else if (N < 32768) launch_few<T, true, 2, 4, 3, 64, sizeof(T) == 4 ? 4 : 1>(c);
        else launch_few<T, true, 2, 4, 5, 64, sizeof(T) == 4 ? 4 : 1>(c);
    }
    else if (K < 2048) launch_few_by_rows<T, 4, 0, 2, 4, 2, 4>(c);
    else if (K >= 16384 && N >= 8192) launch_few_by_rows<T, 8, 64, 4, 2, 4, 2>(c);      // 8192 x 28672 at 16 rows: 80.8 us, in blocks of 16 features 89.9
    else if (half_blocks_for_narrow(N, K)) launch_few_by_rows<T, 8, 64, 1, 5, 1, 4>(c);
    // Blocks of 24 features where they share the weight out more evenly (6144 x 4096 at 8 rows 11.6 us, in blocks of 16 13.5), and from 9 rows on where
    // there are more than two blocks of 16 a unit (10240 x 4096 at 16 rows 20.3, of 16 21.7; at 8 rows 18.8 and 18.1, 14336 x 2048 16.4 and
    // 13.4) -- but not if something is left for a norm, which counts its sums by 16 features.  In bfloat16 the walk along k begins by groups of 48
    // features in all of these: a row's bits depend neither on what is left nor on how many rows there are.  (32-bit, whose bits do
    // differ, keeps groups of 64 and 96: those of 48 cost it 5 % of 5120 x 8192.)
    else if (llmrs_half_tile_blocks(N, 16, cus) || ceil_div(N, 16) > 2 * cus) {
        constexpr int BY16 = sizeof(T) == 2 ? 48 : 64, BY24 = sizeof(T) == 2 ? 48 : 96;
        if (c.next.y != nullptr) launch_few_by_rows<T, 8, BY16, 2, 3, 2, 3>(c);
        else if (ceil_div(N, 16) > 2 * cus && c.M <= 8) launch_few<T, true, 2, 8, 3, BY16, sizeof(T) == 4 ? 4 : 1>(c);
        else launch_few_by_rows<T, 8, BY24, 3, 3, 3, 3>(c);
    }
    else launch_few_by_rows<T, 8, 64, 2, 3, 2, 3>(c);
}

template <class T>
static int gemm_few(hipStream_t stream, const T* A, int lda, const T* W, void* out, int ldc, int M, int N, int K, int epi,
                    const QkvEpilogue* qkv, const RowScale* scale, const NextNorm* next) {
    constexpr int FOUR = 4 * (int)sizeof(T);
    if (scale != nullptr || next != nullptr) {
        bool ok = (scale == nullptr || (scale->sumsq != nullptr && scale->nparts >= 1 && scale->eps > 0.0f)) &&
                  (next == nullptr || (epi == LLMRS_EPI_ACCUM_F32 && llmrs_gemm_leaves_norm(N) && next->sumsq != nullptr && next->y != nullptr &&
                                       next->weight != nullptr && next->ldy >= N && next->ldy % 4 == 0 && (uintptr_t)next->y % FOUR == 0));
        if (!ok) { llmrs_fail("gemm: a deferred norm is taken for up to 16 rows (what is left for the next one: with the += epilogue, a multiple of 4 and under 16384 features), got M=%d N=%d K=%d epilogue %d", M, N, K, epi); return -1; }
    }
    if (epi == LLMRS_EPI_QKV && (M > 16 || qkv == nullptr || !llmrs_qkv_by_fours(qkv->head_dim, qkv->rotary_dim) || ldc % 4 || (uintptr_t)out % FOUR || (uintptr_t)qkv->k_cache % FOUR))
        return 0;
    few_rows<T>(FewCall{stream, A, lda, W, out, ldc, M, N, K, epi, qkv ? *qkv : QkvEpilogue{}, scale ? *scale : RowScale{}, next ? *next : NextNorm{}});
    return 1;
}
int llmrs_gemm_few_bf16(hipStream_t stream, const bf16* A, int lda, const bf16* W, void* out, int ldc, int M, int N, int K, int epi,
                        const QkvEpilogue* qkv, const RowScale* scale, const NextNorm* next) {
    return gemm_few<bf16>(stream, A, lda, W, out, ldc, M, N, K, epi, qkv, scale, next);
}
int llmrs_gemm_few_f32(hipStream_t stream, const float* A, int lda, const float* W, void* out, int ldc, int M, int N, int K, int epi,
                       const QkvEpilogue* qkv, const RowScale* scale, const NextNorm* next) {
    return gemm_few<float>(stream, A, lda, W, out, ldc, M, N, K, epi, qkv, scale, next);
}

// ---- products of a recurrent mixer's single tokens, with what the mixer does with their sums (FewConv, FewGru, FewScan) ------------
// bfloat16, up to 16 requests; the rest is for the product and the kernels of recurrent.hip.
template <int NG, int NW, int R, int ROT, class Extra>
static void launch_mixer_step(const FewCall& c, const Extra& extra) {
    if (c.M <= 8) with_few_launcher<bf16, true, NG, NW, R, ROT>(c, [&](auto launch) { launch(extra); });
    else with_few_launcher<bf16, false, NG, NW, R, ROT>(c, [&](auto launch) { launch(extra); });
}
static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
static bool step_rows_ok(const void* A, int lda, const void* W, int M, int K, const float* state, long state_stride, const int* slots) {
    return M >= 0 && M <= 16 && K > 0 && K % 8 == 0 && lda >= K && lda % 8 == 0 && aligned16(A) && aligned16(W) && state != nullptr && aligned16(state) &&
           state_stride % 4 == 0 && slots != nullptr;
}

// sums = A W^T, of which the first C columns go through the causal convolution of four taps [C, 4] and silu into x (bfloat16) and into the state
// [slots][3][C], and the others, C to N, to out (32-bit, row stride ldc, its first C columns left as they are).
extern "C" int llmrs_conv_product_step(hipStream_t stream, const bf16* A, int lda, const bf16* W, int M, int N, int K, float* out, int ldc, const float* taps,
                                       const float* bias, float* state, long state_stride, const int* slots, int C, bf16* x, int ldx) {
    LLMRS_REQUIRE(step_rows_ok(A, lda, W, M, K, state, state_stride, slots) && state_stride >= 3L * C, "conv_product_step: bad rows or state, M=%d K=%d", M, K);
    LLMRS_REQUIRE(C > 0 && C % 4 == 0 && N >= C && N % 4 == 0 && ldc >= N && ldc % 4 == 0 && ldx >= C && ldx % 4 == 0 && aligned16(out) && aligned16(taps) &&
                  aligned16(bias) && taps != nullptr && ((uintptr_t)x & 7) == 0, "conv_product_step: bad sizes N=%d C=%d", N, C);
    if (M == 0) return 0;
    FewCall c{stream, A, lda, W, out, ldc, M, N, K, LLMRS_EPI_STORE_F32, QkvEpilogue{}, RowScale{}, NextNorm{}};
    FewConv e{taps, bias, state, state_stride, slots, x, ldx, C};
    // (as the plain product's rule above: few rows of a weight, many, and short ones.  The widest, product and kernel -> here, us: up to 8 rows rings of
    // four where the plain product takes seven tiles, of three elsewhere (8 rows 20480 x 5120 41.7 -> 40.0, with three 43.3; 16384 x 4096 27.8 -> 24.9,
    // with four 26.2); a few rows more rings of four (11 rows 18432 x 4608 42.8 -> 34.4, in blocks of 32
    // features 37.4), and beyond, or over the very widest, blocks of twice as many features, which read the rows half as often (16 rows 24576 x 6144
    // 58.8 -> 56.8, 62.0 in blocks of 16; 32768 x 8192 96.3 -> 92.6 and 103; 12 rows 24576 x 6144 in blocks of 16 59.3).)
    if (N >= 16384) {
        if (M <= 8 && wide_tiles(N, llmrs_compute_units()) != 7) launch_mixer_step<2, 4, 3, 64>(c, e);
        else if (M <= (N >= 32768 ? 8 : N >= 22528 ? 10 : 12)) launch_mixer_step<2, 4, 4, 64>(c, e);
        else launch_mixer_step<4, 4, 3, 64>(c, e);
    }
    else if (K < 2048) launch_mixer_step<2, 4, 4, 0>(c, e);
    else if (half_blocks_for_narrow(N, K)) launch_mixer_step<1, 8, 4, 64>(c, e);
    else launch_mixer_step<2, 8, 3, 64>(c, e);
    LLMRS_LAUNCH_CHECK("conv_product_step");
    return 0;
}
// W: [3 width, K], the rows of gate, candidate and output gate; out: [M, width] bfloat16; state [slots][width].
extern "C" int llmrs_mingru_product_step(hipStream_t stream, const bf16* A, int lda, const bf16* W, int M, int width, int K, const float* bias_z, const float* bias_c,
                                         float* state, long state_stride, const int* slots, bf16* out, int ldo) {
    LLMRS_REQUIRE(step_rows_ok(A, lda, W, M, K, state, state_stride, slots) && state_stride >= width, "mingru_product_step: bad rows or state, M=%d K=%d", M, K);
    LLMRS_REQUIRE(width > 0 && width % 8 == 0 && ldo >= width && ldo % 4 == 0 && ((uintptr_t)out & 7) == 0 && aligned16(bias_z) && aligned16(bias_c),
                  "mingru_product_step: bad sizes, width %d", width);
    if (M == 0) return 0;
    // A unit's LDS holds one block of eight waves with rings of three.  With more blocks than units, blocks of four waves share a unit: two with rings of
    // four, three with rings of three (from 9 rows on, and where three a unit are one round of a weight whose rows are short) or two (rows of less than 2048,
    // which fill no deeper one).  (Product and kernel, eight waves, four, us: 4 rows 2560 x 2560 12.2, 14.4, 12.3; 4096 x 4096 21.8, 22.4, 20.0; 5632 x
    // 5632 39.6, 38.7, 35.1; 5120 x 2560 18.5, 21.8, 17.7, with rings of four 19.0; 8192 x 1024 14.1, -, 13.0, with rings of four 14.7; 16 rows 2560 x 2560
    // 15.2, 15.5, 13.5; up to 256 blocks 4 rows 2048 x 2048 9.5, 7.9, 8.0.  Product and kernel stay ahead for two to six rows of 5120 x 5120, 31.2 and
    // 32.3, and for widths of twenty rows' length, 10240 x 512 11.1 and 11.9.)
    const FewCall call{stream, A, lda, W, out, ldo, M, 3 * width, K, LLMRS_EPI_STORE, QkvEpilogue{}, RowScale{}, NextNorm{}};
    const FewGru step{bias_z, bias_c, state, state_stride, slots};
    const int blocks = width / 8, cus = llmrs_compute_units();
    if (blocks <= cus) launch_mixer_step<3, 8, 3, 48>(call, step);
    else if (blocks > 2 * cus && K < 2048) launch_mixer_step<3, 4, 2, 48>(call, step);
    else if (M <= 8 && !(blocks > 2 * cus && blocks <= 3 * cus && K < 4096)) launch_mixer_step<3, 4, 4, 48>(call, step);
    else launch_mixer_step<3, 4, 3, 48>(call, step);
    LLMRS_LAUNCH_CHECK("mingru_product_step");
    return 0;
}
// dt = d Wdt^T (d: [M, K], W: [C, K]), and the selective scan's step of 16 states with it.  x [M, C], b and c [M, 16] (16-byte aligned rows, ldbc apart),
// out [M, C] bfloat16; A [16, C] negative, D [C], gate [M, C] 32-bit; state [slots][16][C].
extern "C" int llmrs_scan_product_step(hipStream_t stream, const bf16* d, int ldd, const bf16* W, int M, int C, int K, const float* dt_bias, const float* A,
                                       const float* D, const float* gate, int ld_gate, float* state, long state_stride, const int* slots, const bf16* x, int ldx,
                                       const bf16* b, const bf16* c, int ldbc, bf16* out, int ldo) {
    LLMRS_REQUIRE(step_rows_ok(d, ldd, W, M, K, state, state_stride, slots) && state_stride >= 16L * C, "scan_product_step: bad rows or state, M=%d K=%d", M, K);
    LLMRS_REQUIRE(C > 0 && C % 16 == 0 && A && D && gate && x && out && ld_gate >= C && ldx >= C && ldo >= C && ldbc >= 16 && ldbc % 8 == 0 && b && c && aligned16(b) &&
                  aligned16(c), "scan_product_step: bad sizes, C=%d", C);
    if (M == 0) return 0;
    // (rings of two k-blocks: a rank of up to 512 is no more than that to a wave, and deeper rings keep blocks off a unit, which wait for the
    // state's bytes here: 9 rows 10240 x 320 9.8 -> 8.4 us, 16384 x 512 at 4 10.0 -> 7.9)
    launch_mixer_step<2, 4, 2, 0>(FewCall{stream, d, ldd, W, out, ldo, M, C, K, LLMRS_EPI_STORE, QkvEpilogue{}, RowScale{}, NextNorm{}},
                                  FewScan{dt_bias, A, D, gate, state, state_stride, slots, x, b, c, ld_gate, ldx, ldbc});
    LLMRS_LAUNCH_CHECK("scan_product_step");
    return 0;
}
