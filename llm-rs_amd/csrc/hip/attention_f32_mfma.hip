// Causal attention of prompt portions in true 32-bit on the matrix cores:
// v_mfma_f32_32x32x2_f32 multiplies and adds in 32-bit (no reduced-precision mode),
// softmax in 32-bit as everywhere, probabilities never rounded.  It takes the place of the
// one-wave-per-token walk of attention_generic.hip for entries with several tokens when
// the engine computes in float32: a 2,048-token prompt is then bound by its products again.
//
// One wave owns 32 columns (the heads of one kv head for a few consecutive tokens of one
// request; four waves may share them, a quarter of the keys each) and walks the keys it may see in tiles of 32, aligned to absolute positions:
//   S^T[key][col] = sum_d K[key][d] Q[col][d]        A operand = keys' rows, B = queries' rows
//   online softmax down each column (a lane holds 16 of a column's 32 keys, its partner
//   in the other half of the wave the other 16)
//   O^T[d][col] += sum_key V[key][d] P[key][col]      A = values, B = the probabilities where they stand
// An MFMA contracts two values, one from each half of the wave; which two is free as long as
// both operands agree.  For QK^T step (j, c) contracts d = 8j + c (lower half) and 8j + 4 + c
// (upper half), so a lane reads its row four consecutive values at a time; for PV step s
// contracts the two keys whose probabilities the two halves hold in register s of S^T, so the
// probabilities feed the second product without moving.  Values lie transposed in the cache,
// [feature][slot], so a lane reads four consecutive keys of its feature at a time.
// A distance penalty with the distance itself is these kernels' (one with its logarithm is left to the walk).
// Needs head_dim % 32 == 0 (up to 256), page_size % 4 == 0, at most 32 heads per kv head,
// 16-byte aligned rows; otherwise the caller keeps to the walk.
// Entries with one token are shared out over waves by key range on the same products (attn_f32_split_kernel): a
// decode step in 32-bit reads its keys and values once for all heads of a kv head, 16 bytes a lane.
// Differential attention (MAPS 2): neighbouring columns are the two maps of a head, c even the first; a column's query is
// zero in the other map's features, and the columns' results are made one at the end (or by the merge).
// Formulas: shaders/ops.metal:636-758 (scale after the dot, causal bound, softmax, weighted sum).
#include "attention.h"
#include "cache_layout.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float swap_halves(float x) {
    unsigned u = __float_as_uint(x);
    auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float((threadIdx.x & 32) ? sw[0] : sw[1]);
}

// One wave's walk over the keys [t_begin, t_end) (t_begin a multiple of 32) for its 32 columns: column c of this lane
// sees the keys lo..pos (pos < 0: a column that is not there).  Adds to the running maximum m (base 2, scale applied),
// the sum l and the sums O^T as they stand.
template <int HD>
__device__ __forceinline__ void f32_walk(const f32x4 (&qf)[HD / 8], const float* __restrict__ kc, const float* __restrict__ vc,
                                         const int* __restrict__ table, const AttnArgs& a, int kvh, int c, int h, int pos, int lo, const AttnFar& far,
                                         int t_begin, int t_end, f32x16 (&O)[HD / 32], float& m, float& l) {
    const int ps = a.page_size;
    const float log2e = 1.44269504088896341f;
    const float scale_log2e = a.scale * log2e;                    // exponentials in base 2: one multiply-add and one v_exp_f32
    const bool capped = a.softcap > 0.0f;                         // scores bent into (-cap, cap) first
    const float inv_cap = capped ? 1.0f / a.softcap : 0.0f, cap_log2e = a.softcap * log2e;
    const int keep = a.keep_first;                                // first keys that stay visible when the window has passed them
    auto page_of = [&](int key) {
        int pg = table[min(key / ps, a.table_width - 1)];
        return min(max(pg, 0), a.num_pages - 1);                   // stay inside the cache whatever the table holds
    };
    for (int t0 = t_begin; t0 < t_end; t0 += 32) {
        // the key this lane's A-operand row holds, and its row in the cache
        int key = t0 + c;
        const float* kp = kc + k_cache_index(page_of(key), kvh, key % ps, 4 * h, a.n_kv_heads, ps, HD);
        f32x4 kf[HD / 8];
#pragma unroll
        for (int j = 0; j < HD / 8; ++j) kf[j] = *(const f32x4*)(kp + 8 * j);
        // the values this lane's A-operand rows hold: feature dt * 32 + c, keys t0 + 8 g + 4 h .. + 3, g = 0..3.
        // Head sizes up to 128: all asked for now, so that their trip runs beside the first product; larger ones
        // (whose registers would not hold them all) one 32-feature tile at a time, right before its product.
        constexpr bool V_AHEAD = HD <= 128;
        const float* vp[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            int k0 = t0 + 8 * g + 4 * h;
            vp[g] = vc + v_cache_index(page_of(k0), kvh, k0 % ps, c, a.n_kv_heads, ps, HD);
        }
        f32x4 vf[V_AHEAD ? HD / 32 : 1][4];
        if constexpr (V_AHEAD) {
#pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
                for (int g = 0; g < 4; ++g) vf[dt][g] = *(const f32x4*)(vp[g] + (size_t)dt * 32 * ps);
        }
        f32x16 S;
#pragma unroll
        for (int i = 0; i < 16; ++i) S[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < HD / 8; ++j)
#pragma unroll
            for (int cc = 0; cc < 4; ++cc) S = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j][cc], qf[j][cc], S, 0, 0, 0);
        // register i of S holds the dot of this lane's column with key t0 + 8 (i / 4) + 4 h + i % 4
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            int kk = t0 + 8 * (i >> 2) + 4 * h + (i & 3);
            float sc = capped ? cap_log2e * tanhf(S[i] * a.scale * inv_cap) : S[i] * scale_log2e;
            if (far.kind) sc = fmaf(-far.r1, (float)(pos - kk), sc);      // (kind 2: r1 has log2 e in it)
            S[i] = (kk > pos || (kk < lo && kk >= keep)) ? -INFINITY : sc;
            mx = fmaxf(mx, S[i]);
        }
        mx = fmaxf(mx, swap_halves(mx));
        float m_new = fmaxf(m, mx);
        float m_safe = m_new == -INFINITY ? 0.0f : m_new;          // a column that has seen no key yet
        float alpha = __builtin_amdgcn_exp2f(m - m_safe);          // (-inf - x: 0)
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            S[i] = __builtin_amdgcn_exp2f(S[i] - m_safe);
            sum += S[i];
        }
        sum += swap_halves(sum);
        l = l * alpha + sum;
        m = m_new;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) O[dt][i] *= alpha;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt) {
            if constexpr (!V_AHEAD) {
#pragma unroll
                for (int g = 0; g < 4; ++g) vf[0][g] = *(const f32x4*)(vp[g] + (size_t)dt * 32 * ps);
            }
#pragma unroll
            for (int s = 0; s < 16; ++s)
                O[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[V_AHEAD ? dt : 0][s >> 2][s & 3], S[s], O[dt], 0, 0, 0);
        }
    }
}

// Values 8j + 4h .. 8j + 4h + 3 of the query at `qp` (which points 4h into its row), those of the map's own features.
template <int HD, int MAPS>
__device__ __forceinline__ void f32_query(f32x4 (&qf)[HD / 8], const float* qp, int map) {
#pragma unroll
    for (int j = 0; j < HD / 8; ++j) {
        qf[j] = *(const f32x4*)(qp + 8 * j);
        if constexpr (MAPS == 2)
            if ((8 * j >= HD / 2 ? 1 : 0) != map) qf[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
}

// What the waves of a block, each with the same columns and other keys, have come to is made one: the waves after the first leave
// theirs in `others` ([wave - 1][column][HD], ROOM floats a wave) and return false; the first adds them in order to its own
// maximum m (base 2), sum l and sums O, and returns true.
template <int HD, int WAVES, int ROOM>
__device__ __forceinline__ bool f32_meet(f32x16 (&O)[HD / 32], float& m, float& l, float* others, float (*stats)[32][2], int wave, int c, int h, bool cvalid) {
    // a lane holds features dt * 32 + 8 g + 4 h + j of its column
    if (h == 0) { stats[wave][c][0] = m; stats[wave][c][1] = l; }
    if (wave > 0 && cvalid) {
        float* mine = others + (size_t)(wave - 1) * ROOM + c * HD;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(f32x4*)(mine + dt * 32 + 8 * g + 4 * h) = f32x4{O[dt][4 * g], O[dt][4 * g + 1], O[dt][4 * g + 2], O[dt][4 * g + 3]};
    }
    __syncthreads();
    if (wave > 0) return false;
    float top = m, part[WAVES];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, stats[w][c][0]);
    const float safe = top == -INFINITY ? 0.0f : top;                     // (a column that saw no key at all)
    l = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        part[w] = __builtin_amdgcn_exp2f(stats[w][c][0] - safe);            // (-inf - x: 0)
        l = fmaf(stats[w][c][1], part[w], l);
    }
    m = top;
    if (cvalid)
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                f32x4 v[WAVES - 1];
#pragma unroll
                for (int w = 1; w < WAVES; ++w) v[w - 1] = *(const f32x4*)(others + (size_t)(w - 1) * ROOM + c * HD + dt * 32 + 8 * g + 4 * h);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float o = O[dt][4 * g + j] * part[0];
#pragma unroll
                    for (int w = 1; w < WAVES; ++w) o = fmaf(v[w - 1][j], part[w], o);
                    O[dt][4 * g + j] = o;
                }
            }
    return true;
}

// SHARED: a block's four waves have the same columns and a quarter of the keys each, side by side, and meet at the end
// (f32_meet); else four tiles of columns a block, a wave each (and always where the waves' sums would not fit in LDS: head
// sizes over 128).  What bounds either is the longest wave, a trip to memory and 64 MFMAs of 64 cycles (head size 64) for every 32
// keys, where tiles are few; with many the bytes and products.  (A portion of 1023 tokens, 32 heads of 64 on 8 kv heads: a wave to
// a tile 128 us, four 70; which of the two runs: attn_f32_shared.)
template <int HD, int MAPS, bool SHARED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(!SHARED || HD > 96 ? 1 : HD <= 32 ? 4 : HD <= 64 ? 3 : 2))) void attn_f32_tiles_kernel(const float* __restrict__ q, float* __restrict__ out,
                                                             const float* __restrict__ kc, const float* __restrict__ vc,
                                                             const int* __restrict__ block_table,
                                                             const int* __restrict__ positions,
                                                             const int* __restrict__ q_starts, int n_entries,
                                                             AttnArgs a, int G, int tpt, int skip_single) {
    __shared__ float others[SHARED ? 3 * 32 * HD : 1];
    __shared__ float stats[SHARED ? 4 : 1][32][2];
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int c = lane & 31, h = lane >> 5;
    int kvh, tile;
    if constexpr (SHARED) {        // (the last tiles, whose keys are most, first)
        kvh = blockIdx.x % a.n_kv_heads;
        int count = count_tiles(q_starts, n_entries, tpt, skip_single), g = blockIdx.x / a.n_kv_heads;
        if (g >= count) return;
        tile = count - 1 - g;
    } else {
        int task = blockIdx.x * 4 + wave;
        kvh = (task >> 2) % a.n_kv_heads;
        tile = (task / (4 * a.n_kv_heads)) * 4 + (task & 3);
    }
    int e = 0, rem = 0;
    if (!locate_tile(q_starts, n_entries, tpt, skip_single, tile, e, rem)) return;
    int tok0 = q_starts[e] + rem * tpt;
    int ntok = min(tpt, q_starts[e + 1] - tok0);
    int tq = c / G, hg = c - tq * G;
    bool cvalid = tq < ntok;
    int token = tok0 + min(tq, ntok - 1);
    int head = (kvh * G + hg) / MAPS;              // (G: columns of a kv head)
    int pos = cvalid ? positions[token] : -1;
    int lo = attn_window_lo(a, pos);
    int last = positions[tok0 + ntok - 1], first = positions[tok0];
    int t_end = last + 1;
    int t_begin = attn_window_lo(a, first) & ~31;
    const int* table = block_table + (size_t)e * a.table_width;

    // this lane's part of its column's query: values 8j + 4h .. 8j + 4h + 3
    f32x4 qf[HD / 8];
    f32_query<HD, MAPS>(qf, q + (size_t)token * a.q_stride + (size_t)head * HD + 4 * h, c % MAPS);
    f32x16 O[HD / 32];
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[dt][i] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    const AttnFar far = attn_far_base2(a, head);
    // the first keys that stay visible, where they lie before the tiles of the window (those among the window's tiles
    // pass the mask there)
    if (a.keep_first > 0 && t_begin > 0 && (!SHARED || wave == 0)) f32_walk<HD>(qf, kc, vc, table, a, kvh, c, h, pos, lo, far, 0, min(a.keep_first, t_begin), O, m, l);
    if constexpr (SHARED) {
        int each = ((t_end - t_begin + 127) >> 7) * 32, from = t_begin + wave * each;
        f32_walk<HD>(qf, kc, vc, table, a, kvh, c, h, pos, lo, far, from, min(from + each, t_end), O, m, l);
        if (!f32_meet<HD, 4, 32 * HD>(O, m, l, others, stats, wave, c, h, cvalid)) return;
    } else f32_walk<HD>(qf, kc, vc, table, a, kvh, c, h, pos, lo, far, t_begin, t_end, O, m, l);
    float inv = 1.0f / (l + attn_sink_term_base2(a, head, m));      // (the sum is complete here: the sink joins it once)
    if constexpr (MAPS == 2) {
        float ss = 0.0f;
#pragma unroll
        for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float mine = O[dt][i] * inv, other = __shfl_xor(mine, 1, 64);      // the column beside this one is the head's other map
                float o = (c & 1) ? other - a.diff_lambda * mine : mine - a.diff_lambda * other;
                O[dt][i] = o;
                ss = fmaf(o, o, ss);
            }
        ss += swap_halves(ss);
        inv = 1.0f / sqrtf(ss / (float)HD + a.diff_eps) * a.diff_scale;
    }
    if (!cvalid || c % MAPS) return;
    float* op = out + (size_t)token * a.out_stride + (size_t)head * HD + 4 * h;
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = O[dt][4 * g + j] * inv * attn_gate(a, token, head, 4 * h + dt * 32 + 8 * g + j);
            *(f32x4*)(op + dt * 32 + 8 * g) = v;
        }
}

// Entries with one token: a block for each (entry, kv head, chunk of F32_SPLIT_CHUNK keys, aligned to absolute positions):
// its columns are the heads of the kv head (the other columns of the 32 multiply zeros: the keys and values are read
// once for all of them, 16 bytes a lane).  It leaves what the walk of
// attention_generic.hip leaves for such a chunk, where that file's merge finds it: the maximum (natural logarithm's
// scale), the sum and the weighted values of each head, [entry][head][chunk][2 + head_dim].
// WAVES 4: each wave takes 32 of the chunk's keys, and the waves' results are added in order through LDS.  With few blocks what
// bounds this step is neither bytes nor products but a wave's chain (a trip to memory, then 64 to 256 MFMAs of 64 cycles, for
// every 32 keys one after the other): four waves side by side take a quarter of it (8 requests of 200 to 1800 keys, 8 kv heads
// of 64: 27.9 -> 21.8 us with the merge; 4 of 1800 keys, heads of 128: 43 -> 37).  WAVES 1, one wave for all of the chunk's
// keys: where blocks are many, or the columns' sums would not fit in LDS (attn_f32_split_four).
template <int HD, int MAPS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(WAVES == 1 || HD > 96 ? 1 : HD <= 32 ? 4 : HD <= 64 ? 3 : 2))) void attn_f32_split_kernel(const float* __restrict__ q, float* __restrict__ partial,
                                                            const float* __restrict__ kc, const float* __restrict__ vc,
                                                            const int* __restrict__ block_table,
                                                            const int* __restrict__ q_starts, const int* __restrict__ seq_lens,
                                                            int max_chunks, AttnArgs a, int G) {
    static_assert(WAVES == 1 || WAVES * 32 == F32_SPLIT_CHUNK, "a wave for every 32 keys of a chunk, or one for all");
    __shared__ float others[WAVES > 1 ? (WAVES - 1) * 2048 : 1];              // [wave - 1][column][HD]
    __shared__ float stats[WAVES][32][2];                                      // [wave][column]: maximum (base 2), sum
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 31, h = lane >> 5;
    int kvh = WAVES > 1 ? blockIdx.x : blockIdx.y, e = WAVES > 1 ? blockIdx.y : blockIdx.x, ch = blockIdx.z;      // (see the launcher)
    int token = q_starts[e];
    if (q_starts[e + 1] - token != 1) return;
    int pos_t = seq_lens[e] - 1;                  // an entry with one token: its position is its length less one
    int lo = attn_window_lo(a, pos_t);
    int first = lo / F32_SPLIT_CHUNK;
    if (ch > pos_t / F32_SPLIT_CHUNK - first) return;                         // (the same for all of a block's waves)
    int begin = max(lo, (first + ch) * F32_SPLIT_CHUNK), end = min(pos_t + 1, (first + ch + 1) * F32_SPLIT_CHUNK);
    bool cvalid = c < G;
    int column = kvh * G + min(c, G - 1), head = column / MAPS;         // (G: columns of a kv head; see the partial results' layout)
    int pos = cvalid ? pos_t : -1;
    const int* table = block_table + (size_t)e * a.table_width;
    f32x4 qf[HD / 8];
    f32_query<HD, MAPS>(qf, q + (size_t)token * a.q_stride + (size_t)head * HD + 4 * h, c % MAPS);
    f32x16 O[HD / 32];
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) O[dt][i] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    const AttnFar far = attn_far_base2(a, head);
    if (wave == 0 && ch == 0 && a.keep_first > 0 && (begin & ~31) > 0)      // the first chunk's (first) wave also takes the kept first keys
        f32_walk<HD>(qf, kc, vc, table, a, kvh, c, h, pos, lo, far, 0, min(a.keep_first, begin & ~31), O, m, l);
    if constexpr (WAVES == 1) f32_walk<HD>(qf, kc, vc, table, a, kvh, c, h, pos, lo, far, begin & ~31, end, O, m, l);
    else {
        int from = (first + ch) * F32_SPLIT_CHUNK + 32 * wave;
        f32_walk<HD>(qf, kc, vc, table, a, kvh, c, h, pos, lo, far, max(from, begin & ~31), min(from + 32, end), O, m, l);
        if (!f32_meet<HD, WAVES, 2048>(O, m, l, others, stats, wave, c, h, cvalid)) return;
    }
    if (!cvalid) return;
    float* pp = partial + ((size_t)(e * a.n_heads * MAPS + column) * max_chunks + ch) * (HD + 2);
    if (h == 0) { pp[0] = m * 0.69314718055994531f; pp[1] = l; }
    // this lane holds features dt * 32 + 8 g + 4 h + j of its column (rows of 2 + head_dim floats: 8-byte aligned)
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
                float2 v = make_float2(O[dt][4 * g + j], O[dt][4 * g + j + 1]);
                *(float2*)(pp + 2 + dt * 32 + 8 * g + 4 * h + j) = v;
            }
}

// Whether four waves share a tile's keys, by `tiles` waves to a SIMD with a wave to a tile, and `reach`, how many keys a tile may
// see.  With 32 keys or fewer three of the four would have none.  Measured, shared against a wave to a tile (1 to 128 portions of
// 2 to 2048 tokens, at positions 0 to 2000): heads of 32 0.26-0.99 everywhere else; heads of 64, 96 and 128: 0.76-0.90 up to a
// quarter of a wave and 64 keys (1.0-2.5 with more tiles); 0.40-0.93 up to half a wave and 256 keys (0.6-1.7 with more);
// 0.30-0.9 up to one wave and any keys (heads of 128: three quarters; at one wave up to 1.1).  With more tiles than that the waves
// of a device are even enough alone: heads of 128 0.9-1.3 unless the portions are long (512 tokens and more: 0.61-1.02), of 64
// and 96 0.6-0.93 over 1100 keys, up to 1.13 under.
static bool attn_f32_shared(int hd, double tiles, int reach, bool long_portions) {
    if (hd > 128 || reach <= 32) return false;
    if (hd <= 32) return true;
    if (tiles <= (reach <= 64 ? 0.25 : reach <= 256 ? 0.5 : hd <= 96 ? 1.0 : 0.75)) return true;
    return reach > 256 && (long_portions || (hd <= 96 && reach > 1100));
}

// Takes the entries with several tokens (all entries when skip_single is 0).  max_seq_len, n_single: what the host knows of the
// entries (an upper bound of their lengths, how many bring one token), or 0 and -1.  Returns 1 when it took them,
// 0 when the shape is not its own (the caller then walks), -1 on error.
int llmrs_attention_f32_mfma(hipStream_t stream, const float* q, float* out, const float* k_cache, const float* v_cache,
                             const int* block_table, const int* positions, const int* q_starts, int n_entries,
                             int skip_single, int max_seq_len, int n_single, const AttnArgs& a) {
    int G = a.n_heads / a.n_kv_heads * a.maps;
    if (a.v_dim != a.head_dim || (a.dist_r1 != nullptr && a.dist_r2 != nullptr)) return 0;
    if (a.head_dim % 32 || a.head_dim > 256 || a.page_size % 4 || G > 32 || q_starts == nullptr) return 0;
    if (a.q_stride % 4 || a.out_stride % 4 || ((uintptr_t)q & 15) || ((uintptr_t)out & 15) || ((uintptr_t)k_cache & 15) ||
        ((uintptr_t)v_cache & 15))
        return 0;
    int tpt = 32 / G;
    long tiles = a.n_tokens / tpt + n_entries;
    // The bound on the lengths holds for single tokens too, whose caches may be longer than the portions': beside them (or where
    // the host does not say) a portion reaches as many keys as it has tokens, at least.
    const int alone = skip_single && n_single > 0 ? min(n_single, n_entries - 1) : 0, mean = (a.n_tokens - alone) / max(1, n_entries - alone);
    int reach = n_single == 0 && max_seq_len > 0 ? max_seq_len : mean;
    if (a.window > 0) reach = min(reach, a.window + tpt + 31 + a.keep_first);
    if (a.mask_chunk > 0) reach = min(reach, a.mask_chunk);
    const double waves = (double)(a.n_tokens / tpt + n_entries) * a.n_kv_heads / (4.0 * llmrs_compute_units());
    const bool shared = attn_f32_shared(a.head_dim, waves, reach, mean >= 512);
    long blocks = (shared ? tiles : (tiles + 3) / 4) * a.n_kv_heads;
    if (blocks > 0x7fffffffL) return 0;
    switch (a.head_dim) {
#define TILES_(HD, MM, SS) attn_f32_tiles_kernel<HD, MM, SS><<<(int)blocks, 256, 0, stream>>>(q, out, k_cache, v_cache, block_table, positions, q_starts, n_entries, a, G, tpt, skip_single)
#define TILES(HD, MM) do { if (shared) TILES_(HD, MM, (HD <= 128)); else TILES_(HD, MM, false); } while (0)
#define CASE(HD) case HD: if (a.maps == 2) TILES(HD, 2); else TILES(HD, 1); break;
        CASE(32) CASE(64) CASE(96) CASE(128) CASE(160) CASE(192) CASE(224) CASE(256)
#undef CASE
#undef TILES
#undef TILES_
        default: return 0;
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        llmrs_fail("attention (32-bit tiles): launch failed: %s", hipGetErrorString(err));
        return -1;
    }
    return 1;
}

// Whether four waves share a chunk.  A unit holds one such block of heads over 96, two or three of 96 and 64, four of 32, with the
// registers they keep, and their meeting costs what a wave's shorter chain saves once the grid makes several rounds:
// measured, four waves against one (grid in blocks to a unit): heads of 128 0.49-0.84 up to 1.5, 0.51-0.85 at 2, up to 1.07 at
// 3, 1.24-1.91 at 64; of 64 0.53-0.93 up to 3, 0.55-0.94 at 6, up to 1.12 at 8; of 32 up to 0.88 at 6, 1.01 at 11, 1.11 at 16.
// A bound of one chunk may hold 64 keys or fewer, which leaves two of the waves idle: 0.80 up to 1 block to a unit, 1.2-1.3 at
// 1.5 to 4.  Counted over the grid, which a recorded step keeps, not over the keys of the moment.
static bool attn_f32_split_four(int columns, int hd, long blocks, int max_chunks) {
    const long to_a_unit = max_chunks == 1 ? 1 : hd <= 32 ? 12 : hd <= 96 ? 6 : 2;
    return columns * hd <= 2048 && blocks <= to_a_unit * llmrs_compute_units();
}

// Takes the entries with one token, split by key range into `partial` (max_chunks chunks of F32_SPLIT_CHUNK keys an
// entry; the caller merges them).  Returns 1 when it took them, 0 when the shape is not its own, -1 on error.
int llmrs_attention_f32_mfma_split(hipStream_t stream, const float* q, float* partial, const float* k_cache, const float* v_cache,
                                   const int* block_table, const int* q_starts, const int* seq_lens, int n_entries,
                                   int max_chunks, const AttnArgs& a) {
    int G = a.n_heads / a.n_kv_heads * a.maps;
    if (a.v_dim != a.head_dim || (a.dist_r1 != nullptr && a.dist_r2 != nullptr)) return 0;
    if (a.head_dim % 32 || a.head_dim > 256 || a.page_size % 4 || G > 32 || q_starts == nullptr || seq_lens == nullptr) return 0;
    if (a.q_stride % 4 || ((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15) || ((uintptr_t)partial & 7))
        return 0;
    if (n_entries > 65535 || a.n_kv_heads > 65535 || max_chunks > 65535 || max_chunks < 1) return 0;
    const bool four = attn_f32_split_four(G, a.head_dim, (long)a.n_kv_heads * n_entries * max_chunks, max_chunks);
    // The chunk last, as short and empty ones are an entry's last (32 requests of 200 keys under a bound of 1024, 8 kv heads of 64,
    // four waves: 16.6 us, with the chunks before the entries 25).  Blocks go to the XCDs in turn: few blocks with the kv head
    // first, so that every XCD gets a share of every entry; many with the entry first, as a first dimension of a few
    // blocks hands thousands of empty ones out more slowly (64 requests of 200 keys under 8192, heads of 128: 47 against 51 us).
    dim3 grid(four ? a.n_kv_heads : n_entries, four ? n_entries : a.n_kv_heads, max_chunks);
    switch (a.head_dim) {
#define SPLIT(HD, MM, WW) attn_f32_split_kernel<HD, MM, WW><<<grid, 64 * WW, 0, stream>>>(q, partial, k_cache, v_cache, block_table, q_starts, seq_lens, max_chunks, a, G)
#define CASE(HD) case HD: if (four) { if (a.maps == 2) SPLIT(HD, 2, 4); else SPLIT(HD, 1, 4); } \
                          else { if (a.maps == 2) SPLIT(HD, 2, 1); else SPLIT(HD, 1, 1); } break;
        CASE(32) CASE(64) CASE(96) CASE(128) CASE(160) CASE(192) CASE(224) CASE(256)
#undef CASE
#undef SPLIT
        default: return 0;
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        llmrs_fail("attention (32-bit split): launch failed: %s", hipGetErrorString(err));
        return -1;
    }
    return 1;
}
