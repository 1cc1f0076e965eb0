// A residual stream that is held in 32-bit whatever the model's compute type: RMS norm with the pieces that
// stand around it (a gate in front, a gain stored around zero or around one, groups of a row normalised apart,
// a residual that the scaled result is added to), the weighted sum of the streams that earlier layers left,
// and the small conversions between the 32-bit stream and the compute type.
//
// Every sum over a row is taken in 32-bit in an order that depends on the row's length alone, so a token's
// values do not depend on what else is in the step.
#include "common.h"
#include "pta_kernels.h"

// v = x (* silu(gate)); n = v / sqrt(mean_group(v^2) + eps) * (offset + w); out = residual + mult * n (or n).
// With `planes` the result (in out_wide) is the last of `count` streams that lie `plane` floats apart, and the launch
// goes on to their weighted sum (mix_wide, and out_narrow in the compute type), as depth_mix_kernel forms it.
// One workgroup per (row, group).  TI: type of x (float or the compute type), T: compute type (gate, narrow output).
template <typename TI, typename T>
__global__ void rmsnorm_kernel(T* __restrict__ out_narrow, float* __restrict__ out_wide, const TI* __restrict__ x,
                               long x_ld, const T* __restrict__ gate, long gate_ld, const int* __restrict__ rows,
                               const float* __restrict__ w, float offset, int group_len, float eps,
                               const float* __restrict__ residual, float mult, int H,
                               const float* __restrict__ planes, long plane, const float* __restrict__ coef, int count,
                               float* __restrict__ mix_wide) {
    __shared__ float red[16];
    const int m = blockIdx.x, g = blockIdx.y;
    const long src = rows ? rows[m] : m;
    const TI* xr = x + src * x_ld + (long)g * group_len;
    const T* gr = gate ? gate + src * gate_ld + (long)g * group_len : nullptr;
    float ss = 0.f;
    for (int i = threadIdx.x; i < group_len; i += blockDim.x) {
        float v = Io<TI>::ld(xr + i);
        if (gr) { const float z = Io<T>::ld(gr + i); v *= z / (1.0f + expf(-z)); }
        ss += v * v;
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)group_len + eps);
    const long o = (long)m * H + (long)g * group_len;
    for (int i = threadIdx.x; i < group_len; i += blockDim.x) {
        float v = Io<TI>::ld(xr + i);
        if (gr) { const float z = Io<T>::ld(gr + i); v *= z / (1.0f + expf(-z)); }
        float n = v * inv * (offset + w[g * group_len + i]);
        if (residual) n = residual[src * H + (long)g * group_len + i] + mult * n;
        if (out_wide) out_wide[o + i] = n;
        if (planes) {  // the result is the last of `count` streams: what goes on is their weighted sum, added in order
            float acc = 0.f;
#pragma unroll 8
            for (int j = 0; j + 1 < count; ++j) acc += coef[j] * planes[(long)j * plane + o + i];
            n = acc + coef[count - 1] * n;
            mix_wide[o + i] = n;
        }
        if (out_narrow) Io<T>::st(out_narrow + o + i, n);
    }
}

// The same for groups of at most VPT * blockDim elements: a thread keeps its VPT elements in registers between the
// two passes, and every pass asks for all of its loads before it uses one (a row of a few thousand elements in a
// step of a few rows is a chain of memory round trips and nothing else).
template <typename TI, typename T, int VPT>
__global__ void rmsnorm_reg_kernel(T* __restrict__ out_narrow, float* __restrict__ out_wide, const TI* __restrict__ x,
                                   long x_ld, const T* __restrict__ gate, long gate_ld, const int* __restrict__ rows,
                                   const float* __restrict__ w, float offset, int group_len, float eps,
                                   const float* __restrict__ residual, float mult, int H,
                                   const float* __restrict__ planes, long plane, const float* __restrict__ coef, int count,
                                   float* __restrict__ mix_wide) {
    __shared__ float red[16];
    const int m = blockIdx.x, g = blockIdx.y;
    const long src = rows ? rows[m] : m;
    const TI* xr = x + src * x_ld + (long)g * group_len;
    const T* gr = gate ? gate + src * gate_ld + (long)g * group_len : nullptr;
    float v[VPT], z[VPT];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        const int i = threadIdx.x + k * blockDim.x;
        v[k] = i < group_len ? Io<TI>::ld(xr + i) : 0.f;
        z[k] = (gr && i < group_len) ? Io<T>::ld(gr + i) : 0.f;
    }
    const long o = (long)m * H + (long)g * group_len;
    float wv[VPT], rv[VPT];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {  // asked for now, used after the sum
        const int i = threadIdx.x + k * blockDim.x;
        wv[k] = i < group_len ? w[g * group_len + i] : 0.f;
        rv[k] = (residual && i < group_len) ? residual[src * H + (long)g * group_len + i] : 0.f;
    }
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        if (gr) v[k] *= z[k] / (1.0f + expf(-z[k]));
        ss += v[k] * v[k];
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)group_len + eps);
    float n[VPT];
#pragma unroll
    for (int k = 0; k < VPT; ++k) {
        n[k] = v[k] * inv * (offset + wv[k]);
        if (residual) n[k] = rv[k] + mult * n[k];
    }
    if (out_wide) {
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            if (i < group_len) out_wide[o + i] = n[k];
        }
    }
    if (planes) {
        float acc[VPT];
#pragma unroll
        for (int k = 0; k < VPT; ++k) acc[k] = 0.f;
        for (int j = 0; j + 1 < count; ++j) {
            const float c = coef[j];
            const float* pj = planes + (long)j * plane + o;
            float pv[VPT];
#pragma unroll
            for (int k = 0; k < VPT; ++k) {
                const int i = threadIdx.x + k * blockDim.x;
                pv[k] = i < group_len ? pj[i] : 0.f;
            }
#pragma unroll
            for (int k = 0; k < VPT; ++k) acc[k] += c * pv[k];
        }
        const float c = coef[count - 1];
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            n[k] = acc[k] + c * n[k];
            if (i < group_len) mix_wide[o + i] = n[k];
        }
    }
    if (out_narrow) {
#pragma unroll
        for (int k = 0; k < VPT; ++k) {
            const int i = threadIdx.x + k * blockDim.x;
            if (i < group_len) Io<T>::st(out_narrow + o + i, n[k]);
        }
    }
}

// four neighbouring elements, loaded and stored at once
__device__ __forceinline__ void ld4(const float* p, float (&v)[4]) {
    const float4 q = *reinterpret_cast<const float4*>(p);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
}
__device__ __forceinline__ void ld4(const bf16_t* p, float (&v)[4]) {
    const uint2 q = *reinterpret_cast<const uint2*>(p);
    v[0] = bf16_bits_to_f32((bf16_t)(q.x & 0xffffu)); v[1] = bf16_bits_to_f32((bf16_t)(q.x >> 16));
    v[2] = bf16_bits_to_f32((bf16_t)(q.y & 0xffffu)); v[3] = bf16_bits_to_f32((bf16_t)(q.y >> 16));
}
__device__ __forceinline__ void st4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ void st4(bf16_t* p, const float (&v)[4]) {
    *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16),
                                              (uint32_t)f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16));
}

// four neighbouring elements as they lie in memory: what is widened where it is loaded is waited for at the next branch, with all before it
template <typename T> struct Raw4;
template <> struct Raw4<float> {
    float4 q;
    __device__ __forceinline__ void load(const float* p) { q = *reinterpret_cast<const float4*>(p); }
    __device__ __forceinline__ void widen(float (&v)[4]) const { v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w; }
};
template <> struct Raw4<bf16_t> {
    uint2 q;
    __device__ __forceinline__ void load(const bf16_t* p) { q = *reinterpret_cast<const uint2*>(p); }
    __device__ __forceinline__ void widen(float (&v)[4]) const {
        v[0] = bf16_bits_to_f32((bf16_t)(q.x & 0xffffu)); v[1] = bf16_bits_to_f32((bf16_t)(q.x >> 16));
        v[2] = bf16_bits_to_f32((bf16_t)(q.y & 0xffffu)); v[3] = bf16_bits_to_f32((bf16_t)(q.y >> 16));
    }
};

// The same where rows can be read four elements at a time (C times four a thread, at most 8,192 a group).  In a step of a
// few rows the launch is one chain (load, sum over the workgroup, store) and its length is instructions as much as trips to
// memory: 2,048 features of 8 rows 3.4 -> 2.4 us (with a gate 4.5 -> 2.9); of 2,000 rows 9.5 -> 6.0 us.
// What the loads are found by comes first and packed, in the fourteen words that are in registers when a workgroup starts; the others are a load away.
// sizes: a group's elements, | planes << 16, | 1 << 30 with a gate, | 1 << 31 where rows are picked.  MIX > 0: a sum of streams is wanted, and its first MIX
// planes (fewer: the last again, so that the wait for the row counts the loads behind it) are asked for with the row.  Behind the norm they came one
// after the other: 8 rows of 2,048 with 2 / 5 / 9 planes 2.70, 3.05, 3.07 -> 2.54, 2.65, 3.02 us over warm caches; 192 such norms of a request, half of them with
// planes, 9.00 -> 8.87 ms.
#define MOST_PLANES 255

template <typename TI, typename T, int C, int MIX>
__global__ __launch_bounds__(1024) void rmsnorm_vec_kernel(
    const TI* __restrict__ x, const float* __restrict__ w, const float* __restrict__ residual, const float* __restrict__ planes,
    const float* __restrict__ coef, uint32_t x_ld, uint32_t plane, int H, uint32_t sizes, const T* __restrict__ gate, long gate_ld,
    const int* __restrict__ rows, T* __restrict__ out_narrow, float* __restrict__ out_wide, float* __restrict__ mix_wide, float offset, float eps, float mult) {
    __shared__ float red[16];
    const int m = blockIdx.x, g = blockIdx.y, group_len = sizes & 0xffff, before = MIX ? (int)(sizes >> 16 & 0xff) - 1 : 0;
    const int threads = ((group_len / 4 + 63) / 64 * 64 / C + 63) / 64 * 64;
    const bool gated = sizes >> 30 & 1;
    long src = m;
    if (sizes >> 31) {
        asm volatile("");
        src = rows[m];
    }
    const TI* xr = x + src * x_ld + (long)g * group_len;
    const float* wr = w + (long)g * group_len;
    const float* rr = residual ? residual + src * H + (long)g * group_len : nullptr;
    const long o = (long)m * H + (long)g * group_len;
    constexpr int AHEAD = MIX ? MIX : 1;
    float v[C][4], cf[AHEAD];
    Raw4<TI> xq[C];
    Raw4<T> gq[C];
    Raw4<float> wq[C], rq[C], pq[C][AHEAD];
#pragma unroll
    for (int c = 0; c < C; ++c) {  // (a thread past the group's end reads its start)
        const int i = 4 * (threadIdx.x + c * threads), at = i < group_len ? i : 0;
        xq[c].load(xr + at);
        wq[c].load(wr + at);
        if (rr) rq[c].load(rr + at);
        if (gated) {
            asm volatile("");
            gq[c].load(gate + src * gate_ld + (long)g * group_len + at);
        }
#pragma unroll
        for (int j = 0; j < MIX; ++j) pq[c][j].load(planes + (long)max(min(j, before - 1), 0) * plane + o + at);
    }
#pragma unroll
    for (int j = 0; j < MIX; ++j) cf[j] = coef[min(j, before)];
    float own = MIX ? coef[before] : 0.f;
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::"s"(out_narrow), "s"(out_wide), "s"(mix_wide), "s"(offset), "s"(eps), "s"(mult));  // asked for here, not where they are used
    if constexpr (MIX > 0) {
        asm volatile("" : "+s"(own));
#pragma unroll
        for (int j = 0; j < MIX; ++j) asm volatile("" : "+s"(cf[j]));
    }
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const bool in = 4 * ((int)threadIdx.x + c * threads) < group_len;
        xq[c].widen(v[c]);
        if (gated) {
            float z[4];
            gq[c].widen(z);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[c][e] *= z[e] / (1.0f + expf(-z[e]));
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[c][e] = in ? v[c][e] : 0.f;
        ss += (v[c][0] * v[c][0] + v[c][1] * v[c][1]) + (v[c][2] * v[c][2] + v[c][3] * v[c][3]);
    }
    ss = block_sum(ss, red, threads / 64);
    const float inv = 1.0f / sqrtf(ss / (float)group_len + eps);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int i = 4 * (threadIdx.x + c * threads);
        if (i >= group_len) continue;
        float n[4], wv[4], rv[4];
        wq[c].widen(wv);
        if (rr) rq[c].widen(rv);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            n[e] = v[c][e] * inv * (offset + wv[e]);
            if (rr) n[e] = rv[e] + mult * n[e];
        }
        if (out_wide) st4(out_wide + o + i, n);
        if constexpr (MIX > 0) {
            float acc[4] = {0.f, 0.f, 0.f, 0.f}, pv[4];
#pragma unroll
            for (int j = 0; j < AHEAD; ++j)
                if (j < before) {
                    pq[c][j].widen(pv);
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[e] += cf[j] * pv[e];
                }
            for (int j = AHEAD; j < before; ++j) {
                ld4(planes + (long)j * plane + o + i, pv);
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] += coef[j] * pv[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) n[e] = acc[e] + own * n[e];
            st4(mix_wide + o + i, n);
        }
        if (out_narrow) st4(out_narrow + o + i, n);
    }
}

extern "C" int pta_rmsnorm(void* out_narrow, float* out_wide, const void* x, int x_wide, long x_ld, const void* gate,
                           long gate_ld, const int* rows, const float* w, float offset, int groups, float eps,
                           const float* residual, float mult, const float* planes, long plane, const float* coef,
                           int count, float* mix_wide, int M, int H, int dtype, void* stream) {
    PTA_REQUIRE(M > 0 && H > 0, "rmsnorm: M=%d H=%d must be positive", M, H);
    PTA_REQUIRE(x && w && (out_narrow || out_wide), "rmsnorm: null pointer");
    PTA_REQUIRE(groups > 0 && H % groups == 0, "rmsnorm: %d features do not split into %d equal groups", H, groups);
    PTA_REQUIRE(groups <= 65535, "rmsnorm: at most 65535 groups, got %d", groups);
    PTA_REQUIRE(x_ld >= H && (!gate || gate_ld >= H), "rmsnorm: rows lie closer together than they are long");
    PTA_REQUIRE(dtype == PTA_F32 || dtype == PTA_BF16, "rmsnorm: unknown dtype %d", dtype);
    PTA_REQUIRE(!planes || (coef && count >= 1 && mix_wide && out_wide && !rows && plane >= (long)M * H),
                "rmsnorm: a sum of streams needs their weights, the planes' distance and both 32-bit results");
    hipStream_t s = (hipStream_t)stream;
    const int L = H / groups;
    const dim3 grid(M, groups), block(L >= 2048 ? 512 : L > 64 ? 256 : 64);
#define RMS_ARGS(TN, TX, TG) (TN*)out_narrow, out_wide, (const TX*)x, x_ld, (const TG*)gate, gate_ld, rows, w, offset, L, eps, \
                             residual, mult, H, planes, plane, coef, count, mix_wide
    // Rows, groups and planes start at a multiple of four elements: what every width in use gives.  Groups below 512 elements
    // are one or two a thread in the kernel for rows that start anywhere and stay there, groups beyond 8,192 take the one that
    // reads its row twice.
    auto on = [](const void* p, size_t bytes) { return (uintptr_t)p % bytes == 0; };
    const size_t narrow = dtype == PTA_F32 ? 16 : 8;
    const bool near = x_ld <= 0xffffffffL && plane <= 0xffffffffL && (!planes || count <= MOST_PLANES);
    if (near && L % 4 == 0 && L >= 512 && L <= 8192 && x_ld % 4 == 0 && (!gate || gate_ld % 4 == 0) && plane % 4 == 0 && on(w, 16) && on(residual, 16) &&
        on(out_wide, 16) && on(planes, 16) && on(mix_wide, 16) && on(gate, narrow) && on(out_narrow, narrow) &&
        on(x, x_wide ? 16 : narrow)) {
        const int threads = (L / 4 + 63) / 64 * 64;
        const uint32_t sizes = (uint32_t)L | (planes ? (uint32_t)count << 16 : 0u) | (gate ? 1u << 30 : 0u) | (rows ? 1u << 31 : 0u);
#define RMS_VEC(TX, T, C, MIX) hipLaunchKernelGGL((rmsnorm_vec_kernel<TX, T, C, MIX>), grid, dim3((threads / C + 63) / 64 * 64), 0, s, (const TX*)x, w, \
                                                  residual, planes, coef, (uint32_t)x_ld, (uint32_t)plane, H, sizes, (const T*)gate, gate_ld, rows, \
                                                  (T*)out_narrow, out_wide, mix_wide, offset, eps, mult)
#define RMS_VEC_C(TX, T) if (threads > 1024) { if (planes) RMS_VEC(TX, T, 2, 2); else RMS_VEC(TX, T, 2, 0); } \
                         else if (!planes) RMS_VEC(TX, T, 1, 0); else if (count <= 3) RMS_VEC(TX, T, 1, 2); \
                         else if (count <= 5) RMS_VEC(TX, T, 1, 4); else RMS_VEC(TX, T, 1, 7)
        if (dtype == PTA_F32) { RMS_VEC_C(float, float); }
        else if (x_wide) { RMS_VEC_C(float, bf16_t); }
        else { RMS_VEC_C(bf16_t, bf16_t); }
#undef RMS_VEC_C
#undef RMS_VEC
        return pta_check_launch("rmsnorm");
    }
    if (L <= 8 * (int)block.x) {  // the group fits the threads' registers
        if (dtype == PTA_F32) hipLaunchKernelGGL((rmsnorm_reg_kernel<float, float, 8>), grid, block, 0, s, RMS_ARGS(float, float, float));
        else if (x_wide) hipLaunchKernelGGL((rmsnorm_reg_kernel<float, bf16_t, 8>), grid, block, 0, s, RMS_ARGS(bf16_t, float, bf16_t));
        else hipLaunchKernelGGL((rmsnorm_reg_kernel<bf16_t, bf16_t, 8>), grid, block, 0, s, RMS_ARGS(bf16_t, bf16_t, bf16_t));
        return pta_check_launch("rmsnorm");
    }
#undef RMS_ARGS
    if (dtype == PTA_F32)
        hipLaunchKernelGGL((rmsnorm_kernel<float, float>), grid, block, 0, s, (float*)out_narrow, out_wide,
                           (const float*)x, x_ld, (const float*)gate, gate_ld, rows, w, offset, L, eps, residual, mult, H, planes, plane, coef, count, mix_wide);
    else if (x_wide)
        hipLaunchKernelGGL((rmsnorm_kernel<float, bf16_t>), grid, block, 0, s, (bf16_t*)out_narrow, out_wide,
                           (const float*)x, x_ld, (const bf16_t*)gate, gate_ld, rows, w, offset, L, eps, residual, mult, H, planes, plane, coef, count, mix_wide);
    else
        hipLaunchKernelGGL((rmsnorm_kernel<bf16_t, bf16_t>), grid, block, 0, s, (bf16_t*)out_narrow, out_wide,
                           (const bf16_t*)x, x_ld, (const bf16_t*)gate, gate_ld, rows, w, offset, L, eps, residual, mult, H, planes, plane, coef, count, mix_wide);
    return pta_check_launch("rmsnorm");
}

// out[i] = sum_j coef[j] * planes[j][i], j = 0 .. count - 1 in that order; the planes lie `plane` floats apart.
template <typename T, int V>
__global__ void depth_mix_kernel(float* __restrict__ out_wide, T* __restrict__ out_narrow,
                                 const float* __restrict__ planes, long plane, const float* __restrict__ coef,
                                 int count, long n) {
    const long i0 = ((long)blockIdx.x * blockDim.x + threadIdx.x) * V;
    if (i0 >= n) return;
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0.f;
    for (int j = 0; j < count; ++j) {
        const float c = coef[j];
        const float* p = planes + (long)j * plane + i0;
        if (V == 4) {
            const float4 q = *reinterpret_cast<const float4*>(p);
            acc[0] += c * q.x; acc[1 % V] += c * q.y; acc[2 % V] += c * q.z; acc[3 % V] += c * q.w;
        } else {
            acc[0] += c * p[0];
        }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        if (out_wide) out_wide[i0 + v] = acc[v];
        if (out_narrow) Io<T>::st(out_narrow + i0 + v, acc[v]);
    }
}

extern "C" int pta_depth_mix(float* out_wide, void* out_narrow, const float* planes, long plane, const float* coef,
                             int count, long n, int dtype, void* stream) {
    PTA_REQUIRE(n > 0 && count > 0, "depth_mix: n=%ld count=%d must be positive", n, count);
    PTA_REQUIRE(planes && coef && (out_wide || out_narrow), "depth_mix: null pointer");
    PTA_REQUIRE(plane >= n, "depth_mix: the planes overlap");
    PTA_REQUIRE(dtype == PTA_F32 || dtype == PTA_BF16, "depth_mix: unknown dtype %d", dtype);
    hipStream_t s = (hipStream_t)stream;
    const bool wide4 = n % 4 == 0 && plane % 4 == 0 && ((uintptr_t)planes % 16) == 0;
    const long threads = wide4 ? n / 4 : n;
    const dim3 grid((unsigned)((threads + 255) / 256)), block(256);
    if (dtype == PTA_F32) {
        if (wide4) hipLaunchKernelGGL((depth_mix_kernel<float, 4>), grid, block, 0, s, out_wide, (float*)out_narrow, planes, plane, coef, count, n);
        else hipLaunchKernelGGL((depth_mix_kernel<float, 1>), grid, block, 0, s, out_wide, (float*)out_narrow, planes, plane, coef, count, n);
    } else {
        if (wide4) hipLaunchKernelGGL((depth_mix_kernel<bf16_t, 4>), grid, block, 0, s, out_wide, (bf16_t*)out_narrow, planes, plane, coef, count, n);
        else hipLaunchKernelGGL((depth_mix_kernel<bf16_t, 1>), grid, block, 0, s, out_wide, (bf16_t*)out_narrow, planes, plane, coef, count, n);
    }
    return pta_check_launch("depth_mix");
}

// out (32-bit) = in (compute type), element by element
template <typename T>
__global__ void widen_kernel(float* __restrict__ out, const T* __restrict__ in, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = Io<T>::ld(in + i);
}

extern "C" int pta_widen(float* out, const void* in, long n, int dtype, void* stream) {
    PTA_REQUIRE(n > 0 && out && in, "widen: nothing to convert");
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
    if (dtype == PTA_F32) hipLaunchKernelGGL(widen_kernel<float>, grid, block, 0, s, out, (const float*)in, n);
    else if (dtype == PTA_BF16) hipLaunchKernelGGL(widen_kernel<bf16_t>, grid, block, 0, s, out, (const bf16_t*)in, n);
    else return pta_fail("widen: unknown dtype %d", dtype);
    return pta_check_launch("widen");
}

__global__ void scale_kernel(float* __restrict__ x, float f, float cap, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = x[i] * f;
    x[i] = cap > 0.f ? cap * tanhf(v / cap) : v;
}

// in place: x *= f, then x = cap tanh(x / cap) where cap > 0 (32-bit)
extern "C" int pta_scale_f32(float* x, float f, float cap, long n, void* stream) {
    PTA_REQUIRE(n > 0 && x, "scale: nothing to scale");
    PTA_REQUIRE(cap >= 0.f, "scale: a cap is positive, or 0 for none");
    hipLaunchKernelGGL(scale_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x, f, cap, n);
    return pta_check_launch("scale");
}
