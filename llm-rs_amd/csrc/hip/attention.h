// Causal attention of a step's query tokens over the paged cache.
#pragma once
#include "common.h"

struct AttnArgs {
    int n_tokens, n_heads, n_kv_heads, head_dim;
    int page_size, table_width, num_pages;
    int q_stride, out_stride;  // elements between tokens
    int window;                // 0: all keys up to the query's position
    float scale;
    int v_dim;                 // width of a value (the cache's values and `out` have it); head_dim where keys and values are alike
    // A penalty that grows with the distance, taken off the scaled (and bent) score of query i and key j, in 32-bit:
    // dist_r1[head] * ln(1 + dist_r2[head] * (i - j)), or with dist_r2 null dist_r1[head] * (i - j).  Both null: none.
    const float* dist_r1;
    const float* dist_r2;
    // > 0: the scaled score s becomes softcap * tanh(s / softcap), in 32-bit, before any penalty and the softmax.
    float softcap;
    // With a window: the first keep_first positions of a request stay visible to every later query, at their true
    // positions.  Key j is visible to the query at i when j <= i and (i - j < window or j < keep_first).
    int keep_first;
    // sink[head], or null: the softmax's denominator of every query of the head also holds exp(sink[head]), once: a key
    // without a value, whose score is this number as it stands (not scaled, not bent, no penalty).
    const float* sink;
    // gate, or null: 32-bit numbers [n_tokens, gate_stride], one for every gate_per consecutive output features of a
    // token (1: a gate a feature; v_dim: a gate a head); the output is multiplied by their sigmoid, in 32-bit, before
    // its one rounding.
    const float* gate;
    int gate_stride, gate_per;
    // > 0 (window 0): positions lie in chunks of so many, counted from the request's position 0, and a query sees the keys
    // of its own chunk only: key j is visible to the query at i when j <= i and j >= i - i % mask_chunk.
    int mask_chunk;
    // 2: differential attention.  A head's row of q and a key's row hold two halves of head_dim / 2 features; each half is
    // an attention (a map) of its own over the same values, and with a1, a2 the maps' results the head's output is
    //   o = a1 - diff_lambda a2,   o / sqrt(mean(o^2) + diff_eps) * diff_scale        (32-bit, before gate and rounding)
    // 1: head_dim features are one map.
    int maps;
    float diff_lambda, diff_eps, diff_scale;
};
// Whether a call is the plain one (values as wide as keys, no distance penalty, no soft cap, no kept first keys) that
// every kernel file takes.
static inline bool attn_is_plain(const AttnArgs& a) {
    return a.v_dim == a.head_dim && a.dist_r1 == nullptr && a.softcap <= 0.0f && (a.keep_first <= 0 || a.window <= 0) && a.sink == nullptr && a.gate == nullptr &&
           a.mask_chunk <= 0 && a.maps == 1;
}
// How many keys a query sees at most (0: all that came before it).
static inline int attn_reach(const AttnArgs& a) { return a.mask_chunk > 0 ? a.mask_chunk : a.window; }
// Chunks of `chunk` keys that a single token's keys can lie in, of `max_chunks` over the whole length.
static inline int attn_chunks_seen(const AttnArgs& a, int max_chunks, int chunk) {
    int reach = attn_reach(a);
    return reach > 0 && (reach - 1) / chunk + 2 < max_chunks ? (reach - 1) / chunk + 2 : max_chunks;
}
// The first key of the window (or the chunk) of the query at `pos`, and how many of the first keys lie before it and
// stay visible.  It never falls as `pos` rises.
__host__ __device__ static inline int attn_window_lo(const AttnArgs& a, int pos) {
    if (a.mask_chunk > 0) return pos > 0 ? pos - pos % a.mask_chunk : 0;
    return (a.window > 0 && pos + 1 > a.window) ? pos + 1 - a.window : 0;
}
__host__ __device__ static inline int attn_kept_before(const AttnArgs& a, int lo) {
    return a.keep_first < lo ? (a.keep_first > 0 ? a.keep_first : 0) : lo;
}

#if defined(__HIPCC__)
// The distance penalty of a head.  kind (the same for all heads): 0 none, 1 with the logarithm of the distance, 2 with
// the distance itself.
struct AttnFar {
    int kind;
    float r1, r2;
};
__device__ __forceinline__ AttnFar attn_far(const AttnArgs& a, int head) {
    if (a.dist_r1 == nullptr) return AttnFar{0, 0.0f, 0.0f};
    if (a.dist_r2 == nullptr) return AttnFar{2, a.dist_r1[head], 0.0f};
    return AttnFar{1, a.dist_r1[head], a.dist_r2[head]};
}
__device__ __forceinline__ float attn_far_term(const AttnFar& f, float distance) {
    return f.kind == 2 ? f.r1 * distance : f.r1 * logf(fmaf(f.r2, distance, 1.0f));
}
// The same for kernels that keep scores in base 2 (times log2 e): r1 ln(.) log2(e) is r1 log2(.), on the hardware's
// logarithm; a penalty with the distance itself has log2(e) in its r1.
__device__ __forceinline__ AttnFar attn_far_base2(const AttnArgs& a, int head) {
    AttnFar f = attn_far(a, head);
    if (f.kind == 2) f.r1 *= 1.4426950408889634f;
    return f;
}
__device__ __forceinline__ float attn_far_term_base2(const AttnFar& f, float distance) {
    return f.kind == 2 ? f.r1 * distance : f.r1 * __builtin_amdgcn_logf(__builtin_fmaf(f.r2, distance, 1.0f));
}
// What the sink of `head` adds to a softmax's sum l whose terms are exp(s - m) (natural: m is a score) or
// 2^(s log2 e - m) (base 2: m is a score times log2 e); 0 without a sink.  Added once, where the sum is complete.
__device__ __forceinline__ float attn_sink_term(const AttnArgs& a, int head, float m) {
    return a.sink ? expf(a.sink[head] - m) : 0.0f;
}
__device__ __forceinline__ float attn_sink_term_base2(const AttnArgs& a, int head, float m2) {
    return a.sink ? __builtin_amdgcn_exp2f(fmaf(a.sink[head], 1.4426950408889634f, -m2)) : 0.0f;
}
// What output feature d of `head` at `token` is multiplied by on its way out: the sigmoid of its gate, or 1.
__device__ __forceinline__ float attn_gate(const AttnArgs& a, int token, int head, int d) {
    if (a.gate == nullptr) return 1.0f;
    float g = a.gate[(size_t)token * a.gate_stride + (head * a.v_dim + d) / a.gate_per];
    return 1.0f / (1.0f + expf(-g));
}
// A step's entries bring their tokens as tiles of `per` tokens that never cross an entry; entries with one token
// bring none when the caller splits those by key range instead.  Which entry holds tile `tile`, and which of that
// entry's tiles it is: a wave finds out together, 64 entries at a time (a serving step has hundreds of entries,
// and a walk from entry to entry by every block cost a prompt portion's kernel more than its own work: 102 ->
// 182 us beside 230 decoding requests).  All lanes of a wave call these with the same arguments and get the same
// answers; false when the tile lies beyond the last one.
__device__ __forceinline__ int tiles_of_entry(const int* __restrict__ q_starts, int n_entries, int i, int per, int skip_single) {
    if (i >= n_entries) return 0;
    int cnt = q_starts[i + 1] - q_starts[i];
    return (cnt == 1 && skip_single) ? 0 : (cnt + per - 1) / per;
}
__device__ __forceinline__ int count_tiles(const int* __restrict__ q_starts, int n_entries, int per, int skip_single) {
    int lane = threadIdx.x & 63, mine = 0;
    for (int i = lane; i < n_entries; i += 64) mine += tiles_of_entry(q_starts, n_entries, i, per, skip_single);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) mine += __shfl_xor(mine, d);
    return mine;
}
__device__ __forceinline__ bool locate_tile(const int* __restrict__ q_starts, int n_entries, int per, int skip_single,
                                            int tile, int& entry, int& within) {
    int lane = threadIdx.x & 63, left = tile;
    for (int base = 0; base < n_entries; base += 64) {
        int nt = tiles_of_entry(q_starts, n_entries, base + lane, per, skip_single);
        int incl = nt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            int v = __shfl_up(incl, d);
            if (lane >= d) incl += v;
        }
        int total = __shfl(incl, 63);
        if (left < total) {
            unsigned long long holds = __ballot(left >= incl - nt && left < incl);    // one lane: its entry has tiles, and this one
            int src = __ffsll((long long)holds) - 1;
            entry = base + src;
            within = left - __shfl(incl - nt, src);
            return true;
        }
        left -= total;
    }
    return false;
}
#endif

// The matrix-core kernels (attention_mfma.hip).  Return 1 when they took the
// call, 0 when its shape is not theirs, -1 on error.
int llmrs_attention_bf16_mfma(hipStream_t stream, const bf16* q, bf16* out, const bf16* k_cache, const bf16* v_cache,
                              const int* block_table, const int* token_entry, const int* positions,
                              const int* q_starts, const int* seq_lens, int n_entries, float* scratch,
                              size_t scratch_bytes, int max_seq_len, int n_single, long single_keys, long portion_keys, const AttnArgs& a);

// Keys per wave when the matrix-core kernels split `singles` single-token entries of up to max_seq_len keys
// that see single_keys keys together (0: unknown; 1 gives the smallest chunk any number of keys can give for these
// entries and this bound, which is what the scratch is sized by).
extern "C" int llmrs_attention_split_chunk(long singles, int n_kv_heads, int head_dim, int max_seq_len, long single_keys);
extern "C" int llmrs_attention_in_shares(int n_tokens, int n_entries, int n_single, long single_keys, long portion_keys, int n_heads, int n_kv_heads, int head_dim,
                                         int reach, int max_seq_len);
extern "C" int llmrs_attention_in_turn(int n_tokens, int n_entries, int n_single, long single_keys, long portion_keys, int n_heads, int n_kv_heads, int head_dim,
                                       int v_dim, int maps);
// How tiles and single tokens go into one grid: the bits say what it does.
#define ATTN_TOGETHER_SHARES 1
#define ATTN_TOGETHER_SINGLES_FIRST 2
extern "C" int llmrs_attention_together(int n_tokens, int n_entries, int n_single, long single_keys, long portion_keys, int n_heads, int n_kv_heads, int head_dim,
                                        int reach, int max_seq_len);

// 32-bit tiles on the matrix cores for entries with several tokens (attention_f32_mfma.hip); skip_single: entries
// with one token are left to the caller.  Return 1 when it took them, 0 when the shape is not its own, -1 on error.
int llmrs_attention_f32_mfma(hipStream_t stream, const float* q, float* out, const float* k_cache, const float* v_cache,
                             const int* block_table, const int* positions, const int* q_starts, int n_entries,
                             int skip_single, int max_seq_len, int n_single, const AttnArgs& a);
// The same for entries with one token, split into chunks of F32_SPLIT_CHUNK keys whose partial results go to `partial`
// in the layout of attention_generic.hip's split, for that file's merge.
#define F32_SPLIT_CHUNK 128
int llmrs_attention_f32_mfma_split(hipStream_t stream, const float* q, float* partial, const float* k_cache, const float* v_cache,
                                   const int* block_table, const int* q_starts, const int* seq_lens, int n_entries,
                                   int max_chunks, const AttnArgs& a);
