// Shared by every kernel file: element types, the error channel of the C
// interface, launch checks.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>

typedef __bf16 bf16;

enum LlmrsDtype { LLMRS_F32 = 0, LLMRS_BF16 = 1 };

// Message of the last failed call on this thread; read through llmrs_hip_error().
char* llmrs_error_buffer();
int llmrs_fail(const char* fmt, ...);
// Compute units of the current device (asked once; 256 if the device cannot be asked).
int llmrs_compute_units();

#define LLMRS_REQUIRE(cond, ...) \
    do {                         \
        if (!(cond)) return llmrs_fail(__VA_ARGS__); \
    } while (0)

#define LLMRS_LAUNCH_CHECK(name)                                              \
    do {                                                                      \
        hipError_t e_ = hipGetLastError();                                    \
        if (e_ != hipSuccess) return llmrs_fail("%s: launch failed: %s", name, hipGetErrorString(e_)); \
    } while (0)

template <class T>
__device__ __forceinline__ float to_f32(T x) { return (float)x; }
template <class T>
__device__ __forceinline__ T from_f32(float x) { return (T)x; }

// Four consecutive elements as 32-bit values: one 16-byte (float) or 8-byte (bfloat16) load.
__device__ __forceinline__ void load4(const float* p, float (&v)[4]) {
    float4 t = *(const float4*)p;
    v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ __forceinline__ void load4(const bf16* p, float (&v)[4]) {
    typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
    bf16x4_t t = *(const bf16x4_t*)p;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (float)t[j];
}

// The sum and the maximum over a wave, all 64 lanes of which must be active, left in every lane.  The moves between lanes are the
// vector unit's own (halves and rows of 16 lanes swapped between registers, then moves within a row: once lanes eight apart agree, a
// turn by four reaches the lane four apart): a few cycles each, where six moves through the LDS crossbar are six trips there, and in
// kernels of one row a block nothing else runs beside them.  Lanes 32, 16, 8, 4, 2 and 1 apart in that order, as a
// butterfly through the crossbar adds them: the same bits.
template <int CTRL, class V>
__device__ __forceinline__ V lanes_moved(V x) {
    return __builtin_bit_cast(V, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}
template <class V, class Op>
__device__ __forceinline__ V wave_fold(V v, Op op) {
    unsigned u = __builtin_bit_cast(unsigned, v);
    auto halves = __builtin_amdgcn_permlane32_swap(u, u, false, false);      // {the low half's, the high half's}
    v = op(__builtin_bit_cast(V, (unsigned)halves[0]), __builtin_bit_cast(V, (unsigned)halves[1]));
    u = __builtin_bit_cast(unsigned, v);
    auto rows = __builtin_amdgcn_permlane16_swap(u, u, false, false);        // {the even row's, the odd row's}
    v = op(__builtin_bit_cast(V, (unsigned)rows[0]), __builtin_bit_cast(V, (unsigned)rows[1]));
    v = op(v, lanes_moved<0x128>(v));            // row_ror:8
    v = op(v, lanes_moved<0x124>(v));            // row_ror:4
    v = op(v, lanes_moved<0x4E>(v));             // quad_perm [2, 3, 0, 1]
    return op(v, lanes_moved<0xB1>(v));          // quad_perm [1, 0, 3, 2]
}
__device__ __forceinline__ float wave_sum(float v) {
    return wave_fold(v, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float wave_max(float v) {
    return wave_fold(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ int wave_min(int v) {
    return wave_fold(v, [](int a, int b) { return min(a, b); });
}

// x / (1 + exp(-x)), as the reference writes it (shaders/ops.metal:769)
__device__ __forceinline__ float silu_f32(float x) { return x / (1.0f + expf(-x)); }

// gelu in its tanh form, x / 2 (1 + tanh(sqrt(2 / pi) (x + 0.044715 x^3))), as x sigmoid(2 sqrt(2 / pi) (x + 0.044715 x^3))
#define GELU_TANH_ALPHA 1.59576912160573071f
#define GELU_TANH_CUBIC 0.044715f
__device__ __forceinline__ float gelu_tanh_f32(float x) { return x / (1.0f + expf(-GELU_TANH_ALPHA * fmaf(GELU_TANH_CUBIC * x * x, x, x))); }

static inline int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }
