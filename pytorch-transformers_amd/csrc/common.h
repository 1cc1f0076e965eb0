// Shared device helpers for the gfx950 kernels: bfloat16 bits, typed loads and
// stores, wave and block reductions, and the error channel of the C entry points.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define PTA_WAVE 64
#define PTA_PAGE 64  // tokens per cache page; must equal cache.paged.PAGE_SIZE

enum PtaDtype { PTA_F32 = 0, PTA_BF16 = 1 };

// orders of the rows of a fused query_key_value projection (described in rope_cache.hip)
enum PtaQkvLayout { PTA_QKV_GROUPED = 0, PTA_QKV_TAIL = 1, PTA_QKV_INTERLEAVED = 2 };

// activations of an epilogue, by the reference's names (src/transformers/activations.py:200-220)
enum PtaAct {
    PTA_ACT_NONE = 0,        // "linear"
    PTA_ACT_GELU = 1,        // "gelu", "gelu_python": the exact erf form
    PTA_ACT_GELU_TANH = 2,   // "gelu_new", "gelu_pytorch_tanh", "gelu_fast", "gelu_accurate"
    PTA_ACT_QUICK_GELU = 3,  // x * sigmoid(1.702 x)
    PTA_ACT_RELU = 4,
    PTA_ACT_RELU2 = 5,       // relu(x)^2
    PTA_ACT_RELU6 = 6,
    PTA_ACT_SILU = 7,        // "silu", "swish"
    PTA_ACT_SIGMOID = 8,
    PTA_ACT_TANH = 9,
    PTA_ACT_LEAKY_RELU = 10, // slope 0.01
    PTA_ACT_MISH = 11,       // x * tanh(softplus(x))
    PTA_ACT_GELU_10 = 12,    // exact GELU clipped to [-10, 10]
    PTA_ACT_LAPLACE = 13,    // the normal distribution function with mean 0.707107, deviation 0.282095
    PTA_ACT_COUNT = 14
};

typedef uint16_t bf16_t;  // raw bits of a bfloat16

__host__ __device__ __forceinline__ float bf16_bits_to_f32(bf16_t v) {
    union { uint32_t u; float f; } c;
    c.u = ((uint32_t)v) << 16;
    return c.f;
}

// round to nearest, ties to even; NaN stays NaN.  On the device this is gfx950's own conversion instruction
// (one for two values where the compiler can pair them); the host spells the same rounding out.
__host__ __device__ __forceinline__ bf16_t f32_to_bf16_bits(float f) {
#if defined(__HIP_DEVICE_COMPILE__)
    union { __bf16 b; bf16_t u; } c;
    c.b = (__bf16)f;
    return c.u;
#else
    union { uint32_t u; float f; } c;
    c.f = f;
    uint32_t u = c.u;
    if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x0040u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (bf16_t)(u >> 16);
#endif
}

__host__ __device__ __forceinline__ float round_to_bf16(float f) { return bf16_bits_to_f32(f32_to_bf16_bits(f)); }

template <typename T> struct Io;
template <> struct Io<float> {
    static __device__ __forceinline__ float ld(const float* p) { return *p; }
    static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
    static __device__ __forceinline__ float round(float v) { return v; }
};
template <> struct Io<bf16_t> {
    static __device__ __forceinline__ float ld(const bf16_t* p) { return bf16_bits_to_f32(*p); }
    static __device__ __forceinline__ void st(bf16_t* p, float v) { *p = f32_to_bf16_bits(v); }
    static __device__ __forceinline__ float round(float v) { return round_to_bf16(v); }
};

// Sums and maxima over lanes, for whole waves.  Between the rows of sixteen lanes by the instructions that exchange halves and rows
// of two registers, within a row by rotated operands: seven instructions in a chain for a wave where __shfl_xor goes through LDS
// six times, each some hundred cycles and a wait.  The additions and their order are those of v + __shfl_xor(v, o) with o as named: a
// rotation by o brings lane i the value of lane i ^ o once those of lanes that are 2 o apart are equal.
struct LaneSum { __device__ __forceinline__ float operator()(float a, float b) const { return a + b; } };
struct LaneMax { __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); } };
template <typename Op> __device__ __forceinline__ float fold_32(float v, Op op) {  // with lane ^ 32
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
template <typename Op> __device__ __forceinline__ float fold_16(float v, Op op) {  // with lane ^ 16
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return op(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
template <int O, typename Op> __device__ __forceinline__ float fold_turned(float v, Op op) {
    return op(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + O, 0xf, 0xf, true)));  // row_ror:O
}
template <typename Op> __device__ __forceinline__ float wave_fold(float v, Op op) {
    v = fold_16(fold_32(v, op), op);
    v = fold_turned<4>(fold_turned<8>(v, op), op);
    return fold_turned<1>(fold_turned<2>(v, op), op);
}
__device__ __forceinline__ float wave_sum(float v) { return wave_fold(v, LaneSum()); }
__device__ __forceinline__ float wave_max(float v) { return wave_fold(v, LaneMax()); }
// over the four lanes that hold a column of a matrix instruction's result
__device__ __forceinline__ float column_sum(float v) { return fold_32(fold_16(v, LaneSum()), LaneSum()); }
__device__ __forceinline__ float column_max(float v) { return fold_32(fold_16(v, LaneMax()), LaneMax()); }

// Sum over a block of up to 1024 threads; every thread gets the result.  `red`
// is LDS of at least 16 floats.  The order of additions depends on the block
// size only.
__device__ __forceinline__ float block_sum(float v, float* red, int nw) {  // nw: the block's waves
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    // all of them asked for at once, what no wave wrote too: a loop of as many as there are waits for LDS in every turn
    float w[16], t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = red[i];
#pragma unroll
    for (int i = 0; i < 16; ++i) t = i < nw ? t + w[i] : t;
    return t;
}
__device__ __forceinline__ float block_sum(float v, float* red) { return block_sum(v, red, (blockDim.x + 63) >> 6); }
__device__ __forceinline__ float block_max(float v, float* red) {
    v = wave_max(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float w[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = red[i];
    float t = w[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) t = i < nw ? fmaxf(t, w[i]) : t;
    return t;
}

// eight bfloat16 in sixteen bytes <-> eight floats
__device__ __forceinline__ void unpack8(const uint4& u, float (&f)[8]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        f[2 * p] = bf16_bits_to_f32((bf16_t)(w[p] & 0xffffu));
        f[2 * p + 1] = bf16_bits_to_f32((bf16_t)(w[p] >> 16));
    }
}
__device__ __forceinline__ uint4 pack8(const float (&f)[8]) {
    typedef __bf16 bf16_pair __attribute__((ext_vector_type(2)));
    typedef float f32_pair __attribute__((ext_vector_type(2)));
    uint32_t w[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        union { bf16_pair b; uint32_t u; } c;
        c.b = __builtin_convertvector(f32_pair{f[2 * p], f[2 * p + 1]}, bf16_pair);  // one instruction for the two
        w[p] = c.u;
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// exact GELU, 0.5 x (1 + erf(x / sqrt 2))  (src/transformers/activations.py:59-78)
__device__ __forceinline__ float gelu_erf(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752440f)); }

// The same for a result that is rounded to bfloat16, in half the instructions: erff works out both of its branches in a wave
// whose lanes differ, some forty instructions an element, which bound the epilogues of large products (a pass over 25,148 x
// 16,384 elements 346 us).  Here x Phi(x) with Phi(-a) = exp(-a^2 / 2) E(a), a = |x|, E fitted as a polynomial of degree eight
// in 1 / (1 + 0.29 a) (the form of Hastings' approximations) to 1.1e-8 of its value up to a = 6 by iterated weighted least
// squares.  Against 64 bits over [-8, 8]: at most 3.8e-7 off, 5.5e-8 in the root mean square, where the erff form is 4.4e-7 and
// 6.2e-8 off; of all finite bfloat16 inputs none is rounded wrongly, by the erff form 188 (below -3, where 1 + erf cancels).
__device__ __forceinline__ float gelu_bf16(float x) {
#pragma clang fp contract(off)  // the last product is not drawn into an addition that follows: the same bits in every epilogue
    const float a = fabsf(x);
    const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(a, 0.29f, 1.0f));
    float p = 0.039498995692840946f;
    p = __builtin_fmaf(p, t, -0.19308443098396097f);
    p = __builtin_fmaf(p, t, 0.30518486352829755f);
    p = __builtin_fmaf(p, t, -0.14805257431489624f);
    p = __builtin_fmaf(p, t, 0.18169167497656202f);
    p = __builtin_fmaf(p, t, 0.07954626252637582f);
    p = __builtin_fmaf(p, t, 0.11979622689254821f);
    p = __builtin_fmaf(p, t, 0.11541898702439371f);
    const float q = p * t * __builtin_amdgcn_exp2f(x * x * -0.72134752044448170368f);  // Phi(-a)
    return x * (x >= 0.f ? 1.0f - q : q);  // an infinity keeps its value above and gives NaN below, as the erff form does
}

// Every activation in 32-bit, rounded once by whoever stores it (src/transformers/activations.py:25-195; softplus
// with torch's threshold of 20, beyond which it is the identity).
__device__ __forceinline__ float apply_act(float x, int act) {
    switch (act) {
        case PTA_ACT_GELU: return gelu_erf(x);
        case PTA_ACT_GELU_TANH: return 0.5f * x * (1.0f + tanhf(0.79788456080286535588f * (x + 0.044715f * x * x * x)));
        case PTA_ACT_QUICK_GELU: return x / (1.0f + expf(-1.702f * x));
        case PTA_ACT_RELU: return fmaxf(x, 0.f);
        case PTA_ACT_RELU2: { const float r = fmaxf(x, 0.f); return r * r; }
        case PTA_ACT_RELU6: return fminf(fmaxf(x, 0.f), 6.f);
        case PTA_ACT_SILU: return x / (1.0f + expf(-x));
        case PTA_ACT_SIGMOID: return 1.0f / (1.0f + expf(-x));
        case PTA_ACT_TANH: return tanhf(x);
        case PTA_ACT_LEAKY_RELU: return x >= 0.f ? x : 0.01f * x;
        case PTA_ACT_MISH: return x * tanhf(x > 20.f ? x : log1pf(expf(x)));
        case PTA_ACT_GELU_10: return fminf(fmaxf(gelu_erf(x), -10.f), 10.f);
        case PTA_ACT_LAPLACE: return 0.5f * (1.0f + erff((x - 0.707107f) / (0.282095f * 1.41421356237309504880f)));
        default: return x;
    }
}

// the same for a result that is rounded to bfloat16
__device__ __forceinline__ float apply_act_bf16(float x, int act) {
#pragma clang fp contract(off)
    if (act == PTA_ACT_GELU) return gelu_bf16(x);
    if (act == PTA_ACT_RELU2) { const float r = fmaxf(x, 0.f); return r * r; }
    return apply_act(x, act);
}

// xIELU with its two coefficients already formed: z > 0: ap z^2 + z / 2; z <= 0: an (e^z - 1 - z) + z / 2
__device__ __forceinline__ float xielu_value(float z, float ap, float an) {
    return z > 0.f ? __builtin_fmaf(ap * z, z, 0.5f * z) : __builtin_fmaf(an, expm1f(z) - z, 0.5f * z);
}

// act(g) * u, or the clamped gate (kinds and fields: PtaGate in pta_kernels.h), in 32-bit
template <typename Gate>
__device__ __forceinline__ float gate_value(float g, float u, int act, const Gate& how) {
    if (how.kind == 1) {
        g = fminf(g, how.limit);
        u = fminf(fmaxf(u, -how.limit), how.limit);
        return g / (1.0f + expf(-how.alpha * g)) * (u + 1.0f);
    }
    return apply_act(g, act) * u;
}

// ---- host side ---------------------------------------------------------
// Entry points return 0 on success; otherwise pta_last_error() holds the reason.
int pta_fail(const char* fmt, ...);
int pta_check_launch(const char* what);
int pta_compute_units();
static inline bool pta_act_known(int act) { return act >= 0 && act < PTA_ACT_COUNT; }

#define PTA_REQUIRE(cond, ...) \
    do { if (!(cond)) return pta_fail(__VA_ARGS__); } while (0)
