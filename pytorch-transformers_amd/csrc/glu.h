// The gate of a feed-forward on a pair of its input product's results, for bfloat16 rows of a multiple of eight elements: the
// gate's own launch (glu_bf16x8_kernel; the clamped kind glu_kernel, with the same expf) and the few-row product's epilogue.
// Rows of other lengths are glu_kernel's, silu with expf and the tanh form with tanhf.
#pragma once

#include "common.h"
#include "pta_kernels.h"

__device__ __forceinline__ float glu_value(int kind, float g, float u, float alpha, float limit) {
    if (kind == PTA_GLU_SILU) return g / (1.0f + __expf(-g)) * u;
    if (kind == PTA_GLU_CLAMPED) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
    }
    // tanh(z) = 1 - 2 / (1 + e^(2z)): both ends saturate without a branch (e^(2z) to infinity or to zero)
    const float z = 0.79788456080286535588f * (g + 0.044715f * g * g * g);
    return g * (1.0f - 1.0f / (1.0f + __expf(2.0f * z))) * u;
}
