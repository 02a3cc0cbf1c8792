// Feed-forwards whose activation runs on a product's 32-bit sums, act(x Wup^T) Wdown^T without a gate projection or
// act(x Wgate^T, x Wup^T) Wdown^T with one, dense or as a mixture of experts.
//
// The router: scores = softmax over all experts of the 32-bit logits; the `top` largest are chosen (of equal scores the
// lower index first); an expert's weight is its score, as it is or divided by the chosen scores' sum.  Or (score kind
// 1) scores = sigmoid(logit) for each expert by itself, chosen by score + correction[e], weighed by the score without
// it (divided by the chosen scores' sum + 1e-20 with `renormalize`), times `scale`.  With `groups` > 1 the experts form so
// many equal groups of neighbours, and only those of the `keep_groups` best groups can be chosen, a group being as good as
// its best expert (by what the choice goes by; of equal groups the lower index first).  The experts' up
// matrices lie one under the other and their down matrices side by side, so that the experts of a token are a dense
// feed-forward of experts * ff hidden units whose activations are multiplied by the expert's weight, zero for the
// experts that were not chosen: the activation kernel below applies act and that weight in one pass.
#include "common.h"

#define ROUTE_MAX_EXPERTS 1024

// The best of a wave's lanes, all of which are active: the largest value, of equal values the lowest index.  (Two folds between
// registers, one for the value and one for the index among the lanes that hold it: both exchanged through the LDS crossbar at
// each of six distances were most of the choice, six of which make up a token's routing.)
__device__ __forceinline__ void wave_best(float& best, int& at) {
    const float most = wave_max(best);
    at = wave_min(best == most ? at : 0x7fffffff);
    best = most;
}

// Takes the experts outside the `keep` best of `groups` groups out of the choice: c[i] (what the choice of expert lane +
// 64 i goes by) becomes `gone` there.  room: 2 ROUTE_MAX_EXPERTS floats of LDS.  All lanes of the block's one wave.
template <int PER>
__device__ __forceinline__ void keep_best_groups(float (&c)[PER], int E, int groups, int keep, float gone, float* room) {
    const int lane = threadIdx.x, per = E / groups;
    float* choice = room;
    float* group = room + ROUTE_MAX_EXPERTS;          // a group's score; once it is kept, what no score is
#pragma unroll
    for (int i = 0; i < PER; ++i)
        if (lane + 64 * i < E) choice[lane + 64 * i] = c[i];
    __syncthreads();
    for (int g = lane; g < groups; g += 64) {
        float best = choice[g * per];
        for (int j = 1; j < per; ++j) best = fmaxf(best, choice[g * per + j]);
        group[g] = best;
    }
    __syncthreads();
    for (int r = 0; r < keep; ++r) {
        float best = -INFINITY;
        int at = 0x7fffffff;
        for (int g = lane; g < groups; g += 64)
            if (group[g] < INFINITY && group[g] > best) { best = group[g]; at = g; }
        wave_best(best, at);
        if (at < groups && (at & 63) == lane) group[at] = INFINITY;
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        if (e < E && group[e / per] < INFINITY) c[i] = gone;
    }
}

// What a shared feed-forward that runs as `shared` further experts behind the E is weighed by: the sigmoid of the number behind
// the experts' logits, the same for all of them.
__device__ __forceinline__ void shared_weights(const float* __restrict__ logits, float* __restrict__ weights, int E, int shared) {
    for (int j = threadIdx.x; j < shared; j += 64) weights[E + j] = 1.0f / (1.0f + expf(-logits[E]));
}

// One wave a token; a lane holds PER experts (E <= 64 PER).  weights [T, E] 32-bit: the chosen experts' weights, zero elsewhere.
template <int PER>
__global__ __launch_bounds__(64) void route_topk_kernel(const float* __restrict__ logits, int ld, float* __restrict__ weights, int ldw,
                                                         int E, int top, int renormalize, int groups, int keep_groups, int shared) {
    __shared__ float room[2 * ROUTE_MAX_EXPERTS];
    int t = blockIdx.x, lane = threadIdx.x;
    float z[PER];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        z[i] = e < E ? logits[(size_t)t * ld + e] : -INFINITY;
        mx = fmaxf(mx, z[i]);
    }
    mx = wave_max(mx);
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        z[i] = (lane + 64 * i) < E ? expf(z[i] - mx) : -1.0f;       // (scores are >= 0: -1 marks what is not there or taken)
        sum += fmaxf(z[i], 0.0f);
    }
    float inv = 1.0f / wave_sum(sum);
    if (groups > 1) keep_best_groups<PER>(z, E, groups, keep_groups, -1.0f, room);
    float keep[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) keep[i] = 0.0f;
    float chosen_sum = 0.0f;
    for (int r = 0; r < top; ++r) {
        float best = -1.0f;
        int at = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (z[i] > best) { best = z[i]; at = lane + 64 * i; }      // ascending index within a lane: the first of equals stays
        wave_best(best, at);
        if (best < 0.0f) break;
        chosen_sum += best * inv;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + 64 * i == at) { keep[i] = z[i] * inv; z[i] = -1.0f; }
    }
    float norm = renormalize ? 1.0f / chosen_sum : 1.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        if (e < E) weights[(size_t)t * ldw + e] = keep[i] * norm;
    }
    shared_weights(logits + (size_t)t * ld, weights + (size_t)t * ldw, E, shared);
}

// Score kind 1.  One wave a token; the chosen experts' weights into weights [T, E], zero elsewhere.
template <int PER>
__global__ __launch_bounds__(64) void route_topk_sigmoid_kernel(const float* __restrict__ logits, int ld, float* __restrict__ weights, int ldw,
                                                                 int E, int top, int renormalize, const float* __restrict__ correction,
                                                                 float scale, int groups, int keep_groups, int shared) {
    __shared__ float room[2 * ROUTE_MAX_EXPERTS];
    int t = blockIdx.x, lane = threadIdx.x;
    float s[PER], c[PER], keep[PER];        // score, what the choice goes by (-inf: not there or taken), the weight kept
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        bool in = e < E;
        s[i] = in ? 1.0f / (1.0f + expf(-logits[(size_t)t * ld + e])) : 0.0f;
        c[i] = in ? s[i] + (correction ? correction[e] : 0.0f) : -INFINITY;
        keep[i] = 0.0f;
    }
    if (groups > 1) keep_best_groups<PER>(c, E, groups, keep_groups, -INFINITY, room);
    float chosen_sum = 0.0f;
    for (int r = 0; r < top; ++r) {
        float best = -INFINITY, best_s = 0.0f;
        int at = 0x7fffffff;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (c[i] > best) { best = c[i]; best_s = s[i]; at = lane + 64 * i; }
        const int own = at;
        wave_best(best, at);
        if (at == 0x7fffffff) break;
        chosen_sum += wave_sum(own == at ? best_s : 0.0f);         // (one lane's: the others add nothing)
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + 64 * i == at) { keep[i] = s[i]; c[i] = -INFINITY; }
    }
    float norm = (renormalize ? 1.0f / (chosen_sum + 1e-20f) : 1.0f) * scale;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int e = lane + 64 * i;
        if (e < E) weights[(size_t)t * ldw + e] = keep[i] * norm;
    }
    shared_weights(logits + (size_t)t * ld, weights + (size_t)t * ldw, E, shared);
}

// score_kind 0: softmax over the experts (correction and scale are not used: null and 1); 1: a sigmoid for each expert,
// chosen by score + correction [E] (null: none), weights times scale.  groups, keep_groups: see above (1, 1: no groups).
// shared: columns of weights behind the experts' that get the sigmoid of logits[t, E] (0: none).
extern "C" int llmrs_route_topk(hipStream_t stream, const float* logits, int ld, float* weights, int ldw, int n_tokens, int E, int top,
                                int renormalize, int score_kind, const float* correction, float scale, int groups, int keep_groups, int shared) {
    LLMRS_REQUIRE(logits && weights && E > 0 && top > 0 && top <= E && shared >= 0 && ld >= E + (shared > 0 ? 1 : 0) && ldw >= E + shared, "route_topk: bad arguments");
    LLMRS_REQUIRE(E <= ROUTE_MAX_EXPERTS, "route_topk: %d experts exceed %d", E, ROUTE_MAX_EXPERTS);
    LLMRS_REQUIRE(score_kind == 0 || score_kind == 1, "route_topk: unknown score kind %d (0: softmax, 1: sigmoid)", score_kind);
    LLMRS_REQUIRE(score_kind == 1 || (correction == nullptr && scale == 1.0f), "route_topk: a correction or a scale goes with sigmoid scores");
    LLMRS_REQUIRE(groups >= 1 && E % groups == 0 && keep_groups >= 1 && keep_groups <= groups, "route_topk: %d experts in %d groups of which %d", E, groups, keep_groups);
    LLMRS_REQUIRE(top <= E / groups * keep_groups, "route_topk: top %d of the %d experts of %d groups", top, E / groups * keep_groups, keep_groups);
    if (n_tokens <= 0) return 0;
#define ROUTE(PER) do { if (score_kind == 1) route_topk_sigmoid_kernel<PER><<<n_tokens, 64, 0, stream>>>(logits, ld, weights, ldw, E, top, renormalize, correction, scale, groups, keep_groups, shared); \
                        else route_topk_kernel<PER><<<n_tokens, 64, 0, stream>>>(logits, ld, weights, ldw, E, top, renormalize, groups, keep_groups, shared); } while (0)
    if (E <= 64) ROUTE(1);
    else if (E <= 256) ROUTE(4);
    else ROUTE(ROUTE_MAX_EXPERTS / 64);
#undef ROUTE
    LLMRS_LAUNCH_CHECK("route_topk");
    return 0;
}

// out[t, c] = act * (weights ? weights[t, c / ff] : 1); up 32-bit sums, out in the activation type (one rounding).
// kind 0: act = relu(up[t, c])^2.  kind 1, a gated activation on sums whose columns are (gate_0, up_0, gate_1, up_1, ...):
// g = min(up[t, 2c], limit), u = clamp(up[t, 2c + 1], -limit, limit), act = g * sigmoid(alpha * g) * (u + 1).
// kind 2, gated, columns as for kind 1: act = silu(gate) * up.  kind 3, gated, likewise: act = gelu(gate) * up in the tanh
// form of gelu, gelu(g) = g sigmoid(2 sqrt(2 / pi) (g + 0.044715 g^3)).
template <class T, int KIND>
__global__ void act_weight_kernel(const float* __restrict__ up, int ldu, const float* __restrict__ weights, int ldw, int ff, int n,
                                  long total, T* __restrict__ out, int ldo, float limit, float alpha) {
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    long t = i / n;
    int c = (int)(i - t * n);
    float y;
    if constexpr (KIND == 0) {
        float x = fmaxf(up[(size_t)t * ldu + c], 0.0f);
        y = x * x;
    } else if constexpr (KIND == 2) {
        float2 gu = *(const float2*)(up + (size_t)t * ldu + 2 * c);
        y = silu_f32(gu.x) * gu.y;
    } else if constexpr (KIND == 3) {
        float2 gu = *(const float2*)(up + (size_t)t * ldu + 2 * c);
        y = gelu_tanh_f32(gu.x) * gu.y;
    } else {
        float2 gu = *(const float2*)(up + (size_t)t * ldu + 2 * c);
        float g = fminf(gu.x, limit), u = fminf(fmaxf(gu.y, -limit), limit);
        y = g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
    }
    if (weights) y *= weights[(size_t)t * ldw + c / ff];
    out[(size_t)t * ldo + c] = from_f32<T>(y);
}

// n: columns of out; up has n columns (kind 0) or 2 n (the others, then ldu even and up 8-byte aligned).
extern "C" int llmrs_act_weight(hipStream_t stream, int dtype, const float* up, int ldu, const float* weights, int ldw, int ff,
                                int n_tokens, int n, int kind, void* out, int ldo, float limit, float alpha) {
    LLMRS_REQUIRE(up && out && n > 0 && ldo >= n && ff > 0 && n % ff == 0, "act_weight: bad arguments");
    LLMRS_REQUIRE(kind >= 0 && kind <= 3, "act_weight: unknown activation %d (0: squared relu, 1: clamped gated sigmoid, 2: gated silu, 3: gated gelu)", kind);
    LLMRS_REQUIRE(ldu >= (kind > 0 ? 2 * n : n), "act_weight: the sums' rows are too short");
    LLMRS_REQUIRE(kind == 0 || (ldu % 2 == 0 && ((uintptr_t)up & 7) == 0), "act_weight: gate and up side by side in 8-byte pairs");
    LLMRS_REQUIRE(kind != 1 || limit > 0.0f, "act_weight: a positive limit");
    LLMRS_REQUIRE(!weights || ldw >= n / ff, "act_weight: the weights' rows are too short");
    long total = (long)n_tokens * n;
    if (total <= 0) return 0;
    LLMRS_REQUIRE(ceil_div(total, 256) <= 0x7fffffff, "act_weight: too many elements for one launch");
    int blocks = ceil_div(total, 256);
#define ACT(TT, KK) act_weight_kernel<TT, KK><<<blocks, 256, 0, stream>>>(up, ldu, weights, ldw, ff, n, total, (TT*)out, ldo, limit, alpha)
    if (dtype == LLMRS_F32) { if (kind == 0) ACT(float, 0); else if (kind == 1) ACT(float, 1); else if (kind == 2) ACT(float, 2); else ACT(float, 3); }
    else if (dtype == LLMRS_BF16) { if (kind == 0) ACT(bf16, 0); else if (kind == 1) ACT(bf16, 1); else if (kind == 2) ACT(bf16, 2); else ACT(bf16, 3); }
    else return llmrs_fail("act_weight: unknown dtype %d", dtype);
#undef ACT
    LLMRS_LAUNCH_CHECK("act_weight");
    return 0;
}

// ---- the experts' rows one after the other --------------------------------------------------------------------------
// For steps of many tokens the chosen (token, expert) pairs are laid out expert by expert, each expert's rows in the
// order of their tokens, so that an expert's tokens are a dense product of their own.  counts[e]: how many tokens chose
// expert e (a block an expert).  With the counts known: row_token[row], row_weight[row] for every row, and
// row_of[t, e] = the row of token t with expert e, or -1 (a block an expert; an expert's first row is the sum of the
// counts before it; each of its four waves takes a quarter of the tokens).
#define ROUTE_ROW_WAVES 4
__device__ __forceinline__ int chosen_in(const float* __restrict__ weights, int ldw, int e, int t_lo, int t_hi) {
    int lane = threadIdx.x & 63, n = 0;
#pragma unroll 4
    for (int t = t_lo + lane; t < t_hi; t += 64) n += weights[(size_t)t * ldw + e] > 0.0f;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) n += __shfl_xor(n, d, 64);
    return n;
}
__global__ __launch_bounds__(64 * ROUTE_ROW_WAVES) void route_counts_kernel(const float* __restrict__ weights, int ldw, int T, int* __restrict__ counts) {
    __shared__ int part[ROUTE_ROW_WAVES];
    int e = blockIdx.x, wave = threadIdx.x >> 6, per = (T + ROUTE_ROW_WAVES - 1) / ROUTE_ROW_WAVES;
    int n = chosen_in(weights, ldw, e, wave * per, min(T, (wave + 1) * per));
    if ((threadIdx.x & 63) == 0) part[wave] = n;
    __syncthreads();
    if (threadIdx.x == 0) counts[e] = part[0] + part[1] + part[2] + part[3];
}

__global__ __launch_bounds__(64 * ROUTE_ROW_WAVES) void route_rows_kernel(const float* __restrict__ weights, int ldw, int T, int E, const int* __restrict__ counts,
                                                         int* __restrict__ row_token, float* __restrict__ row_weight, int* __restrict__ row_of) {
    __shared__ int part[ROUTE_ROW_WAVES];
    int e = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, first = 0;
    int per = (T + ROUTE_ROW_WAVES - 1) / ROUTE_ROW_WAVES, t_lo = wave * per, t_hi = min(T, t_lo + per);
    int mine = chosen_in(weights, ldw, e, t_lo, t_hi);
    if (lane == 0) part[wave] = mine;
    for (int i = lane; i < e; i += 64) first += counts[i];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) first += __shfl_xor(first, d, 64);
    __syncthreads();
    for (int w = 0; w < wave; ++w) first += part[w];
    for (int t0 = t_lo; t0 < t_hi; t0 += 64) {
        int t = t0 + lane;
        float w = t < t_hi ? weights[(size_t)t * ldw + e] : 0.0f;
        unsigned long long chosen = __ballot(w > 0.0f);
        int row = first + __popcll(chosen & ((1ull << lane) - 1ull));
        if (t < t_hi) row_of[(size_t)t * E + e] = w > 0.0f ? row : -1;
        if (w > 0.0f) { row_token[row] = t; row_weight[row] = w; }
        first += __popcll(chosen);
    }
}

extern "C" int llmrs_route_counts(hipStream_t stream, const float* weights, int ldw, int n_tokens, int E, int* counts) {
    LLMRS_REQUIRE(weights && counts && E > 0 && ldw >= E && n_tokens >= 0 && E <= 65535, "route_counts: bad arguments");
    route_counts_kernel<<<E, 64 * ROUTE_ROW_WAVES, 0, stream>>>(weights, ldw, n_tokens, counts);
    LLMRS_LAUNCH_CHECK("route_counts");
    return 0;
}

extern "C" int llmrs_route_rows(hipStream_t stream, const float* weights, int ldw, int n_tokens, int E, const int* counts, int* row_token,
                                float* row_weight, int* row_of) {
    LLMRS_REQUIRE(weights && counts && row_token && row_weight && row_of && E > 0 && ldw >= E && n_tokens >= 0 && E <= 65535, "route_rows: bad arguments");
    route_rows_kernel<<<E, 64 * ROUTE_ROW_WAVES, 0, stream>>>(weights, ldw, n_tokens, E, counts, row_token, row_weight, row_of);
    LLMRS_LAUNCH_CHECK("route_rows");
    return 0;
}

// out[r, :] = x[rows[r], :] (rows of the activation type)
template <class T>
__global__ void gather_rows_kernel(T* __restrict__ out, int ldo, const T* __restrict__ x, int ldx, const int* __restrict__ rows, int D) {
    int r = blockIdx.x, src = rows[r];
    for (int d = threadIdx.x; d < D; d += blockDim.x) out[(size_t)r * ldo + d] = x[(size_t)src * ldx + d];
}

extern "C" int llmrs_gather_rows(hipStream_t stream, int dtype, void* out, int ldo, const void* x, int ldx, const int* rows, int n_rows, int D) {
    LLMRS_REQUIRE(out && x && rows && D > 0 && ldo >= D && ldx >= D && n_rows >= 0, "gather_rows: bad arguments");
    if (n_rows == 0) return 0;
    if (dtype == LLMRS_F32) gather_rows_kernel<float><<<n_rows, 256, 0, stream>>>((float*)out, ldo, (const float*)x, ldx, rows, D);
    else if (dtype == LLMRS_BF16) gather_rows_kernel<bf16><<<n_rows, 256, 0, stream>>>((bf16*)out, ldo, (const bf16*)x, ldx, rows, D);
    else return llmrs_fail("gather_rows: unknown dtype %d", dtype);
    LLMRS_LAUNCH_CHECK("gather_rows");
    return 0;
}

// h[t, :] += sum over the experts e that token t chose, in ascending e, of y[row_of[t, e], :]; 32-bit.  The token's rows are
// listed first; VEC: rows of whole 16-byte pieces.
template <bool VEC>
__global__ __launch_bounds__(256) void combine_rows_kernel(float* __restrict__ h, int ldh, const float* __restrict__ y, int ldy,
                                                           const int* __restrict__ row_of, int E, int D) {
    __shared__ int list[ROUTE_MAX_EXPERTS];
    int t = blockIdx.x, lane = threadIdx.x & 63, n = 0;
    for (int base = 0; base < E; base += 64) {                  // (every wave makes the same list)
        int row = base + lane < E ? row_of[(size_t)t * E + base + lane] : -1;
        unsigned long long has = __ballot(row >= 0);
        if (row >= 0 && threadIdx.x < 64) list[n + __popcll(has & ((1ull << lane) - 1ull))] = row;
        n += __popcll(has);
    }
    __syncthreads();
    if constexpr (VEC) {
        for (int d = 4 * threadIdx.x; d < D; d += 1024) {
            float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
            float4 old = *(const float4*)(h + (size_t)t * ldh + d);
#pragma unroll 4
            for (int i = 0; i < n; ++i) {
                float4 v = *(const float4*)(y + (size_t)list[i] * ldy + d);
                acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
            }
            *(float4*)(h + (size_t)t * ldh + d) = make_float4(old.x + acc.x, old.y + acc.y, old.z + acc.z, old.w + acc.w);
        }
    } else {
        for (int d = threadIdx.x; d < D; d += 256) {
            float acc = 0.0f;
            for (int i = 0; i < n; ++i) acc += y[(size_t)list[i] * ldy + d];
            h[(size_t)t * ldh + d] += acc;
        }
    }
}

extern "C" int llmrs_combine_rows(hipStream_t stream, float* h, int ldh, const float* y, int ldy, const int* row_of, int n_tokens, int E, int D) {
    LLMRS_REQUIRE(h && y && row_of && D > 0 && ldh >= D && ldy >= D && E > 0 && n_tokens >= 0, "combine_rows: bad arguments");
    if (n_tokens == 0) return 0;
    LLMRS_REQUIRE(E <= ROUTE_MAX_EXPERTS, "combine_rows: %d experts exceed %d", E, ROUTE_MAX_EXPERTS);
    bool vec = D % 4 == 0 && ldh % 4 == 0 && ldy % 4 == 0 && ((uintptr_t)h & 15) == 0 && ((uintptr_t)y & 15) == 0;
    if (vec) combine_rows_kernel<true><<<n_tokens, 256, 0, stream>>>(h, ldh, y, ldy, row_of, E, D);
    else combine_rows_kernel<false><<<n_tokens, 256, 0, stream>>>(h, ldh, y, ldy, row_of, E, D);
    LLMRS_LAUNCH_CHECK("combine_rows");
    return 0;
}
