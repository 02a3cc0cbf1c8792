// The matrix-core attention kernels (attention_mfma.h) for heads of one map, what both kinds share, and the rule that
// says by how many keys single tokens are split.
#include "attention_mfma.h"

SideStream* llmrs_attention_side_stream() {
    static SideStream per_device[64];
    static std::mutex mutex;
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    std::lock_guard<std::mutex> lock(mutex);
    SideStream& s = per_device[dev];
    if (!s.tried) {
        s.tried = true;
        bool ok = hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking) == hipSuccess &&
                  hipEventCreateWithFlags(&s.fork, hipEventDisableTiming) == hipSuccess &&
                  hipEventCreateWithFlags(&s.join, hipEventDisableTiming) == hipSuccess;
        if (!ok) { (void)hipGetLastError(); s.stream = nullptr; }
    }
    return s.stream != nullptr ? &s : nullptr;
}

// How many waves of the split a compute unit holds at once: eight (see SPLIT16_LDS_BYTES), fewer where the registers
// of the kernel for this head size allow no more (four at head size 256), asked of the runtime once per head size.
// Head sizes without a kernel here: 8.  (The 32-column kernel, for more than 16 heads to a kv head, holds eight at
// head size 128 as well and twelve at 64; its chunks are chosen as if it held eight.)
static int split_waves_to_a_unit(int head_dim) {
    static int known[8] = {0, 0, 0, 0, 0, 0, 0, 0};      // by head_dim / 32 - 1
    static std::mutex mutex;
    if (head_dim % 32 || head_dim < 32 || head_dim > 256) return 8;
    std::lock_guard<std::mutex> lock(mutex);
    int& n = known[head_dim / 32 - 1];
    if (n == 0) {
        int blocks = 0;
        hipError_t e = hipErrorInvalidValue;
        switch (head_dim) {
#define ASK(HD) case HD: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, attn_split16_kernel<HD, HD, 1>, 64, SPLIT16_LDS_BYTES); break;
            ASK(32) ASK(64) ASK(96) ASK(128) ASK(192) ASK(256)
#undef ASK
            default: break;
        }
        if (e != hipSuccess) (void)hipGetLastError();
        n = (e == hipSuccess && blocks >= 1) ? std::min(blocks, 32) : 8;
    }
    return n;
}

// Keys per wave of the split, by what the host knows: the number of single-token entries, the bound on their
// length, and (when it says so) how many keys they see together.  Measured on the 8B head shape (8 to 256 requests
// of 520 to 8000 keys, every chunk from 64 to 1024 keys) and on the 1B one: a compute unit holds so many of these
// waves at once (eight) and works through them in turns of that many.  Waves of one
// turn, all of the same length, end together, and the longest chunks that still fill half a turn are the fastest
// (a wave begins with a chain of trips to memory: lengths, page numbers, then keys); one wave more than a turn
// costs a second turn.  So: the smallest chunk that gives a unit no more than three quarters of a turn (the next
// length then still gives it more than a third); and when even chunks of 1024
// keys give more than a turn, 512 if the last turn would be far from full (many short waves share out evenly as they come).
// Against the best chunk of each case (also at sizes and lengths between those it was made from, at 4 and 8 heads
// to a kv head, 2 and 8 kv heads) this rule is within the 3 % that two timings of one case differ by, 6 % at worst;
// the rule before the first of this kind (128 keys, doubled while the waves kept all units busy, by the bound alone)
// lost 7.5 % on average and 19 % at worst.  The chunks of a request are never
// more than a quarter of what the merge takes.
// The number of keys moves with every step while a recorded graph holds the chunk it was recorded with: callers that
// record put this function's result into what they key their recordings by.  The scratch is sized by the smallest
// chunk the entries and the bound allow, taken at an eighth of the bound for every entry; fewer keys than that get
// that chunk too.
// LLMRS_SPLIT_CHUNK in the environment (64 to 1024, a power of two) takes the choice away from the rule, for measuring it.
extern "C" int llmrs_attention_split_chunk(long singles, int n_kv_heads, int head_dim, int max_seq_len, long single_keys) {
    if (const char* e = getenv("LLMRS_SPLIT_CHUNK")) {
        int c = atoi(e);
        if (c >= ATTN_CHUNK / 2 && c <= 8 * ATTN_CHUNK && (c & (c - 1)) == 0) return c;
    }
    double cus = (double)llmrs_compute_units();
    if (singles < 1) singles = 1;
    if (max_seq_len < 1) max_seq_len = 1;
    const double turn = split_waves_to_a_unit(head_dim);
    const int longest = 8 * ATTN_CHUNK;
    auto pick = [&](double keys) {
        // waves to a compute unit with chunks of c keys, every entry taken at the mean length; the last chunk of a
        // request counts as a wave unless it is so short that it is gone before it matters
        auto to_a_unit = [&](int c) {
            double q = keys / singles / c, whole = floor(q), rest = q - whole;
            return singles * n_kv_heads * (whole + (rest > 0.125 ? 1.0 : 0.0)) / cus;
        };
        const double full = turn * 1.001;
        // With the 16-column kernel a unit does best on about half a turn of waves, one to a SIMD: a full turn of
        // chunks half as long takes 2-7 % longer, a quarter of a turn of chunks twice as long 15-25 % (8 to 128
        // requests of 520 to 8000 keys, every chunk forced).  So chunks are doubled while a unit would get more than
        // three quarters of a turn: the next length still leaves it more than a third.
        const double enough = 0.75 * turn;
        int c = ATTN_CHUNK / 2;
        while (c < longest && to_a_unit(c) > enough) c *= 2;
        if (c == longest && to_a_unit(c) > full) {
            double last = fmod(to_a_unit(c), turn) / turn;
            if (last > 0.006 && last < 0.69) c /= 2;
        }
        while (c < longest && (max_seq_len + c - 1) / c > MERGE_MAX_CHUNKS / 4) c *= 2;
        return c;
    };
    double bound_keys = (double)singles * max_seq_len;
    int least = pick(bound_keys / 8.0);
    double keys = single_keys > 0 ? fmin((double)single_keys, bound_keys) : 0.75 * bound_keys;
    return std::max(pick(keys), least);
}

// How many keys the tokens of entries with several tokens see together: what the caller says (portion_keys), or, where that is 0, as if
// every such entry began at position 0.
static double keys_of_portions(int n_tokens, int n_entries, int n_single, long portion_keys) {
    const double tokens = n_tokens - n_single;
    return portion_keys > 0 ? (double)portion_keys : tokens * tokens / (2.0 * std::max(n_entries - n_single, 1));
}

// Whether the tiles' blocks are of half as many tokens, in two shares of their keys (attn_tiles_lds_kernel with two shares; one map, heads of up to 128).
// Where there are few blocks the walk of a block along its keys is what takes the time (alone on its unit four waves take 1.17 us a
// tile of 32 keys, and two shares 1.4 for two).  Fuller grids hide one
// block's waits behind another's, and there the second pass over the keys costs more.  us, blocks of four groups and shares, 32 heads on 8:
// 512 tokens over 8512 keys 257 and 139, of 64 features 209 and 117; 128 over 4128 128 and 71; a prompt of 512 24.4 and 18.3, of 1024
// 41 and 30, of 64 features 32 and 21.5; eight of 250 21 and 30; under windows, 400 tokens from 3000 on 44 and 24 (768), 55 and 28 (1024), 1000 tokens 45 and
// 32 (768), 84 and 49 (2048, of 64 features), but 2048 tokens under one of 300 31 and 41; windows in between were not measured.
// With more blocks the longest walk still decides where there are up to 24 blocks for every tile of its keys and little lies before the step's
// tokens (32 heads on 8, 1536 tokens 60 and 49, 1800 from position 100 93 and 60, 2048 78 and 70, of 64 features 60 and 49, prompts of
// 1200 and 300 61 and 36, of 1500 and 500 58 and 50; 40 heads on 5, 1333 tokens 57 and 34; but 64 heads on 8, 1024 tokens
// 46 and 50, twelve prompts of 600 98 and 133, 2048 tokens over 4096 keys 154 and 161).  (blocks: as many as the tokens could make; a prompt or two of 2048
// tokens in all are within the slack of two.)
// Beside single tokens (n_single > 0), whose waves want the units' LDS too, blocks for as many units as their keys leave: all up to 2^25 keys times
// kv heads and features, half up to 68 * 2^20 (64 heads on 8, 200 tokens over 2248 keys beside 4 of 300 115 and 56; 100 over 2148 beside 16 of 4000 120
// and 81; 300 beside 20 of 8000 153 and 168), and a walk that is not over before theirs is, nor within what a step on two streams takes anyway: 25 us and four
// fifths of their keys' time at 5 TB/s.  The walk is taken for the portions' mean place and half their length.  (32 heads on 8, two of 109 tokens from 300 on
// beside 10 of 3200 69.7 and 73.4; 64 on 8, 94 from 300 beside 25 of 2600 72.9 and 77.2; heads of 64, 506 from 300 beside 15 44.0 and 47.9; 230 such steps with
// shares 0.44 to 1.2 of the time, of which the walk's rule leaves 119, 0.44 to 1.05, and four of the others would gain more than 5 %.)
extern "C" int llmrs_attention_in_shares(int n_tokens, int n_entries, int n_single, long single_keys, long portion_keys, int n_heads, int n_kv_heads, int head_dim,
                                         int reach, int max_seq_len) {
    const long cus = llmrs_compute_units(), per_block = 2L * std::max(32 / std::max(n_heads / std::max(n_kv_heads, 1), 1), 1);
    const long blocks = (n_tokens / per_block + n_entries) * n_kv_heads, few = 2 * cus + 2 * n_kv_heads;
    if (max_seq_len < 256 || (reach > 0 && (reach < 768 || blocks > few))) return 0;
    if (n_single <= 0)
        return blocks <= few || (blocks <= 4 * cus + 2 * n_kv_heads && max_seq_len <= n_tokens + n_tokens / 4 && blocks <= 24L * ((max_seq_len + 31) / 32));
    const int tokens = n_tokens - n_single, portions = n_entries - n_single;
    if (tokens <= 0 || portions <= 0 || blocks > 4 * cus) return 0;
    const long busy = (tokens / per_block + portions) * n_kv_heads;
    const long read = (single_keys > 0 ? single_keys : (long)n_single * max_seq_len) * n_kv_heads * head_dim;
    const double walk = keys_of_portions(n_tokens, n_entries, n_single, portion_keys) / tokens + tokens / (2.0 * portions);
    const double walk_us = walk / 32.0 * (head_dim >= 128 ? 1.17 : 0.79), single_us = (double)read * 4.0 / 5e6;
    return busy <= (read <= 1L << 25 ? cus : read <= 68L << 20 ? cus / 2 : 0) && walk_us >= std::max(25.0, 0.8 * single_us);
}

// Whether a mixed step's single tokens wait for its tiles instead of running beside them on a stream of their own.  Their waves that start between two
// rounds of tiles take the LDS that a tile's block of the next round waits for; in turn nothing hides the tiles' last
// round, and the single tokens' keys come when the matrix cores are idle.  So in turn with more than three and three quarters of a block of tiles to a unit (two
// run there at once; 1800 tokens from the start beside 16 of 300, 3.5 of them, 104 and 108) if the single tokens' keys, at 5 TB/s, take no more than a fifth of the tiles' time at 0.7 PFLOP/s.  Measured, us, side by
// side and in turn (64 heads on 8): 2048 tokens from position 2048 beside 16 of 4096 keys, 0.18 of it, 389 and 339; 2940 from 1000 beside 14 of 1300,
// 0.04, 352 and 327; but 1800 from the start beside 16 of 2000, 0.35, 109 and 122; 1600 from 2048 beside 250 of 2000, 1.9, 595 and 619; 32 on 8, 4096
// from 2048 beside 37 of 1500, 0.12, 432 and 383; three of 1365 beside 100 of 2200, 2.8, 262 and 298.  Over 252 steps of
// 1.5 to 8 blocks to a unit, 1 to 256 single tokens and seven shapes of heads what the rule puts in turn takes 0.84 to 1.025 of the time (from
// three blocks on one step would take 1.07); with heads of 64, which need half of the LDS, in turn is 0.92 to 1.48 of it, and the gains are small.
extern "C" int llmrs_attention_in_turn(int n_tokens, int n_entries, int n_single, long single_keys, long portion_keys, int n_heads, int n_kv_heads, int head_dim,
                                       int v_dim, int maps) {
    const int per_tile = 4 * (32 / std::max(n_heads / std::max(n_kv_heads, 1), 1)), portions = n_entries - n_single;
    if (head_dim != 128 || v_dim != 128 || maps != 1 || n_single <= 0 || portions <= 0 || single_keys <= 0 || per_tile == 0) return 0;
    if (((n_tokens - n_single) / per_tile + portions) * (double)n_kv_heads <= 3.75 * llmrs_compute_units()) return 0;
    const double seen = keys_of_portions(n_tokens, n_entries, n_single, portion_keys);
    return (double)single_keys * n_kv_heads * (4.0 * head_dim) / 5e6 <= 0.2 * (seen * n_heads * (4.0 * head_dim) / 0.7e9);
}

// How both kinds of work of a step go into one grid (attn_mixed_kernel): ATTN_TOGETHER_SHARES, the tiles' keys in two shares, where no more than four of their
// blocks come to a unit and their walk is not over well before the single tokens' keys have come (at 5 TB/s); ATTN_TOGETHER_SINGLES_FIRST, the single tokens' first 512
// blocks before the tiles, where their keys take more than 20 us and longer than the tiles' walk.  Of 220 steps (1 to 160 single tokens, one to four
// portions of 2 to 2000 tokens, eight shapes of heads) the time with what the two choose is 1.017 of the best of both choices' six combinations in the mean, and 0.53
// of that on two streams.  Shares, without and with: 32 heads on 8 of 64 features, 23 requests of 445 keys beside a prompt of 1284 58.7 and 38.6; 64 heads on 8,
// 10 of 2300 beside portions of 355 and 453 38.5 and 46.9 (the walk says no), 40 on 8, 4 beside four of 470 45.2 and 52.1 (five blocks to a unit).  Tiles first and single tokens first:
// 64 heads on 8, 68 of 1030 to 1533 beside 1232 tokens 143 and 102; 12 heads of 64, 75 of 1200 beside 98 tokens over 3000 keys (the longer walk) 79 and 98.
extern "C" int llmrs_attention_together(int n_tokens, int n_entries, int n_single, long single_keys, long portion_keys, int n_heads, int n_kv_heads, int head_dim,
                                        int reach, int max_seq_len) {
    const int singles = std::max(n_single, 0), tokens = n_tokens - singles, portions = n_entries - singles;
    if (tokens <= 0 || portions <= 0) return 0;
    const long cus = llmrs_compute_units(), per_block = 2L * std::max(32 / std::max(n_heads / std::max(n_kv_heads, 1), 1), 1);
    const double read = (single_keys > 0 ? (double)single_keys : (double)singles * max_seq_len) * n_kv_heads * head_dim, single_us = read * 4.0 / 5e6;
    double walk = keys_of_portions(n_tokens, n_entries, singles, portion_keys) / tokens + tokens / (2.0 * portions);
    if (reach > 0) walk = std::min(walk, (double)reach);
    const double walk_us = walk / 32.0 * (head_dim >= 128 ? 1.17 : 0.79);
    const bool shares = max_seq_len >= 256 && (reach <= 0 || reach >= 768) && (tokens / per_block + portions) * n_kv_heads <= 4 * cus && walk_us >= 0.25 * single_us;
    return (shares ? ATTN_TOGETHER_SHARES : 0) | (single_us > 20.0 && single_us > walk_us ? ATTN_TOGETHER_SINGLES_FIRST : 0);
}

// Heads of two maps (attention_mfma_maps.hip).
int llmrs_attention_bf16_mfma_maps(hipStream_t stream, const bf16* q, bf16* out, const bf16* k_cache, const bf16* v_cache,
                                   const int* block_table, const int* positions, const int* q_starts, const int* seq_lens,
                                   int n_entries, float* scratch, size_t scratch_bytes, int max_seq_len, int n_single,
                                   long single_keys, long portion_keys, const AttnArgs& a);

int llmrs_attention_bf16_mfma(hipStream_t stream, const bf16* q, bf16* out, const bf16* k_cache, const bf16* v_cache,
                              const int* block_table, const int* token_entry, const int* positions,
                              const int* q_starts, const int* seq_lens, int n_entries, float* scratch,
                              size_t scratch_bytes, int max_seq_len, int n_single, long single_keys, long portion_keys, const AttnArgs& a) {
    (void)token_entry;
    int G = a.n_heads / a.n_kv_heads * a.maps;
    // (a distance penalty is these kernels' too)
    if (a.v_dim != a.head_dim && !(a.maps == 2 && 2 * a.v_dim == a.head_dim)) return 0;
    if (a.maps == 2 && a.v_dim > 256) return 0;
    if (a.keep_first > 1024) return 0;                 // (the tiles of kept first keys: at most 32 a block)
    if (a.page_size != 16 || a.head_dim % 32 || G > 32 || q_starts == nullptr) return 0;
    if (a.q_stride % 8 || a.out_stride % 4 || ((uintptr_t)q & 15) || ((uintptr_t)out & 7)) return 0;
    if (n_entries > 65535 || a.n_kv_heads > 65535) return 0;
    int rc;
    if (a.maps == 2) {
        rc = llmrs_attention_bf16_mfma_maps(stream, q, out, k_cache, v_cache, block_table, positions, q_starts, seq_lens, n_entries,
                                            scratch, scratch_bytes, max_seq_len, n_single, single_keys, portion_keys, a);
        if (rc <= 0) return rc;
    } else switch (a.head_dim) {
#define CASE(HD) case HD: rc = launch<HD, HD, 1>(stream, q, out, k_cache, v_cache, block_table, positions, q_starts, seq_lens, n_entries, scratch, scratch_bytes, max_seq_len, n_single, single_keys, portion_keys, a); break;
        CASE(32) CASE(64) CASE(96) CASE(128) CASE(192) CASE(256)
#undef CASE
        default: return 0;
    }
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) {
        llmrs_fail("attention (mfma): launch failed: %s", hipGetErrorString(err));
        return -1;
    }
    return rc;
}
