// Several residual streams in place of one (hyper-connections), held in 32-bit: per token S vectors x_1 .. x_S.
//
//   x_t <- sum_s mix[s, t] x_s + out[t] * y        (y: what a sublayer left; all streams at once from the old ones)
//   u    = sum_t in[t] x_t                         (what the next sublayer reads; in null: the plain sum)
//   n    = u / sqrt(mean(u^2) + eps) * (offset + w)
//   h    = n + sum_k c[k] * n of K - 1 - k tokens ago   (optional: a causal convolution per channel on the norm's output)
//
// One launch does all of it.  A workgroup owns a token: it forms the new streams feature by feature, leaves u in LDS
// for the second pass, and writes h in the compute type.  The convolution rides in it where every sequence brings one
// token: the inputs from before are then all in the sequence's tail (the last K - 1 norm outputs, oldest first, 32-bit),
// which the same threads move on.  Where sequences bring several tokens the launch leaves n in 32-bit (n_out) for the
// convolution's own launch (pta_conv_add).
#include "common.h"
#include "pta_kernels.h"

#include <algorithm>
#include <type_traits>

#define HYPER_MAX_STREAMS 8

template <int V> struct Vec;
template <> struct Vec<4> {
    static __device__ __forceinline__ void ld(const float* p, float (&v)[4]) {
        const float4 q = *reinterpret_cast<const float4*>(p);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
    }
    static __device__ __forceinline__ void ld(const bf16_t* p, float (&v)[4]) {
        const uint2 q = *reinterpret_cast<const uint2*>(p);
        v[0] = bf16_bits_to_f32((bf16_t)(q.x & 0xffffu)); v[1] = bf16_bits_to_f32((bf16_t)(q.x >> 16));
        v[2] = bf16_bits_to_f32((bf16_t)(q.y & 0xffffu)); v[3] = bf16_bits_to_f32((bf16_t)(q.y >> 16));
    }
    // as it lies in memory: where loads come one behind the other with branches between, words widened at once are waited for at each
    static __device__ __forceinline__ void ld(const float* p, float4& q) { q = *reinterpret_cast<const float4*>(p); }
    static __device__ __forceinline__ void ld(const bf16_t* p, uint2& q) { q = *reinterpret_cast<const uint2*>(p); }
    static __device__ __forceinline__ void widen(const float4& q, float (&v)[4]) { v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w; }
    static __device__ __forceinline__ void widen(const uint2& q, float (&v)[4]) {
        v[0] = bf16_bits_to_f32((bf16_t)(q.x & 0xffffu)); v[1] = bf16_bits_to_f32((bf16_t)(q.x >> 16));
        v[2] = bf16_bits_to_f32((bf16_t)(q.y & 0xffffu)); v[3] = bf16_bits_to_f32((bf16_t)(q.y >> 16));
    }
    static __device__ __forceinline__ void st(float* p, const float (&v)[4]) {
        *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    }
    static __device__ __forceinline__ void st(bf16_t* p, const float (&v)[4]) {
        bf16_t r[4] = {f32_to_bf16_bits(v[0]), f32_to_bf16_bits(v[1]), f32_to_bf16_bits(v[2]), f32_to_bf16_bits(v[3])};
        *reinterpret_cast<uint2*>(p) = make_uint2((uint32_t)r[0] | ((uint32_t)r[1] << 16), (uint32_t)r[2] | ((uint32_t)r[3] << 16));
    }
};
template <> struct Vec<1> {
    template <typename T> static __device__ __forceinline__ void ld(const T* p, float (&v)[1]) { v[0] = Io<T>::ld(p); }
    template <typename T> static __device__ __forceinline__ void ld(const T* p, T& q) { q = *p; }
    template <typename T> static __device__ __forceinline__ void widen(const T& q, float (&v)[1]) { v[0] = Io<T>::ld(&q); }
    template <typename T> static __device__ __forceinline__ void st(T* p, const float (&v)[1]) { Io<T>::st(p, v[0]); }
};

struct HyperArgs {
    void* h;              // [M, H] in the compute type, or null
    float* n_out;         // [M, H], or null
    float* u_out;         // [M, H], or null
    float* x_out;         // [M, S, H], or null
    const float* x;       // row m, stream s at x + m * x_row + s * x_stream
    long x_row, x_stream; // x_stream 0: the streams are all equal, one vector
    const void* y;        // [M, H] rows y_ld apart in the compute type, or null
    long y_ld;
    const float *mix, *out, *in;
    const float* w;
    float offset, eps;
    const int* rows;
    const float* conv;    // [K, H], or null
    int K;
    float* tail;
    long tail_ld;
    const int *token_seq, *seq_slot;
    int H;
};

template <typename T, int S, int V>
__global__ __launch_bounds__(1024) void hyper_norm_kernel(HyperArgs a) {
    extern __shared__ __attribute__((aligned(16))) float u_s[];
    __shared__ float red[16];
    const int m = blockIdx.x, H = a.H;
    const long src = a.rows ? a.rows[m] : m;
    const float* x = a.x + src * a.x_row;
    const T* y = a.y ? (const T*)a.y + src * a.y_ld : nullptr;
    float ss = 0.f;
    for (int i = threadIdx.x * V; i < H; i += blockDim.x * V) {
        float xs[S][V], yv[V], u[V];
#pragma unroll
        for (int s = 0; s < S; ++s) Vec<V>::ld(x + s * a.x_stream + i, xs[s]);
#pragma unroll
        for (int v = 0; v < V; ++v) u[v] = 0.f;
        if (y) Vec<V>::ld(y + i, yv);
#pragma unroll
        for (int t = 0; t < S; ++t) {
            float xt[V];
            if (y) {
                const float o = a.out[t];
#pragma unroll
                for (int v = 0; v < V; ++v) xt[v] = 0.f;
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    const float c = a.mix[s * S + t];
#pragma unroll
                    for (int v = 0; v < V; ++v) xt[v] += c * xs[s][v];
                }
#pragma unroll
                for (int v = 0; v < V; ++v) xt[v] += o * yv[v];
                if (a.x_out) Vec<V>::st(a.x_out + ((long)m * S + t) * H + i, xt);
            } else {
#pragma unroll
                for (int v = 0; v < V; ++v) xt[v] = xs[t][v];
            }
            const float c = a.in ? a.in[t] : 1.f;
#pragma unroll
            for (int v = 0; v < V; ++v) u[v] += c * xt[v];
        }
        Vec<V>::st(u_s + i, u);
        if (a.u_out) Vec<V>::st(a.u_out + (long)m * H + i, u);
#pragma unroll
        for (int v = 0; v < V; ++v) ss += u[v] * u[v];
    }
    if (!a.h && !a.n_out) return;
    const float inv = 1.0f / sqrtf(block_sum(ss, red) / (float)H + a.eps);
    float* tl = a.conv && a.K > 1 ? a.tail + (long)a.seq_slot[a.token_seq[m]] * a.tail_ld : nullptr;
    for (int i = threadIdx.x * V; i < H; i += blockDim.x * V) {
        float n[V], w[V], h[V];
        Vec<V>::ld(u_s + i, n);
        Vec<V>::ld(a.w + i, w);
#pragma unroll
        for (int v = 0; v < V; ++v) n[v] = n[v] * inv * (a.offset + w[v]);
        if (a.n_out) Vec<V>::st(a.n_out + (long)m * H + i, n);
        if (!a.h) continue;
#pragma unroll
        for (int v = 0; v < V; ++v) h[v] = n[v];
        if (a.conv) {
            float acc[V], c[V];
#pragma unroll
            for (int v = 0; v < V; ++v) acc[v] = 0.f;
            for (int k = 0; k + 1 < a.K; ++k) {
                float before[V];
                Vec<V>::ld(tl + (long)k * H + i, before);
                Vec<V>::ld(a.conv + (long)k * H + i, c);
#pragma unroll
                for (int v = 0; v < V; ++v) acc[v] += c[v] * before[v];
                if (k > 0) Vec<V>::st(tl + (long)(k - 1) * H + i, before);  // each input moves one place towards the oldest
            }
            if (a.K > 1) Vec<V>::st(tl + (long)(a.K - 2) * H + i, n);
            Vec<V>::ld(a.conv + (long)(a.K - 1) * H + i, c);
#pragma unroll
            for (int v = 0; v < V; ++v) h[v] += acc[v] + c[v] * n[v];
        }
        Vec<V>::st((T*)a.h + (long)m * H + i, h);
    }
}

// The same where a row has a chunk of V features for each thread of a workgroup (4,096 features) and the convolution up to ONCE_TAPS taps: what every
// published width is.  A step of a few tokens is one chain, and all that does not hang on the norm is asked for at its start: the streams' weights, which the
// loop above loads again behind every store, the norm's, the taps and the sequence's tail, whose row is two look-ups away.  2,048 features, four
// streams, four taps, 2 tokens, in a step: 6.6 us, 5.3 with the loads at the start, 3.6 with none of them behind a wait: a result in 16 bits that is widened where it
// is loaded, a look-up or a weight of the streams that comes by a vector load, an argument that is not there yet each waited for all before it.
#define ONCE_TAPS 4

// What its first loads are found by comes first and packed, in the fourteen words that are in registers when a workgroup starts.  sizes: features | taps
// << 16 | whether rows are picked << 31.
template <typename T, int S, int V>
__global__ __launch_bounds__(1024) void hyper_norm_once_kernel(const float* __restrict__ xs_in, const T* __restrict__ y, const float* __restrict__ norm_w,
                                                               const float* __restrict__ conv, const int* __restrict__ token_seq, uint32_t x_row,
                                                               uint32_t x_stream, uint32_t y_ld, uint32_t sizes, const int* __restrict__ seq_slot,
                                                               const float* __restrict__ mixes, const float* __restrict__ outs, const float* __restrict__ ins,
                                                               const int* __restrict__ rows, HyperArgs a) {
    __shared__ float red[16];
    const int m = blockIdx.x, H = sizes & 0xffff, K = sizes >> 16 & 0xff, waves = max(1, ((H + V - 1) / V + 63) / 64);
    const bool live = (int)threadIdx.x * V < H, normed = norm_w != nullptr;
    const int i = live ? threadIdx.x * V : 0;
    long src = m;
    if (sizes >> 31) {
        asm volatile("");
        src = rows[m];
    }
    float xs[S][V], yv[V], w[V], taps[ONCE_TAPS][V], before[ONCE_TAPS][V];
#pragma unroll
    for (int s = 0; s < S; ++s) Vec<V>::ld(xs_in + src * x_row + (long)s * x_stream + i, xs[s]);
    typename std::conditional<V == 1, T, typename std::conditional<sizeof(T) == 4, float4, uint2>::type>::type yq;
    if (y) Vec<V>::ld(y + src * y_ld + i, yq);
    if (normed) Vec<V>::ld(norm_w + i, w);
    if (conv) {
#pragma unroll
        for (int k = 0; k < ONCE_TAPS; ++k) Vec<V>::ld(conv + (long)min(k, K - 1) * H + i, taps[k]);
    }
    __builtin_amdgcn_sched_barrier(0);
    float mix[S][S], to[S], from[S];
#pragma unroll
    for (int t = 0; t < S; ++t) from[t] = 1.f;
    if (ins) {
#pragma unroll
        for (int t = 0; t < S; ++t) from[t] = ins[t];
    }
    if (y) {
#pragma unroll
        for (int t = 0; t < S; ++t) {
            to[t] = outs[t];
#pragma unroll
            for (int s = 0; s < S; ++s) mix[s][t] = mixes[s * S + t];
        }
    }
    float* tl = conv && K > 1 ? a.tail + (long)seq_slot[token_seq[m]] * a.tail_ld : nullptr;
    if (tl) {
#pragma unroll
        for (int k = 0; k + 1 < ONCE_TAPS; ++k) Vec<V>::ld(tl + (long)min(k, K - 2) * H + i, before[k]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (y) Vec<V>::widen(yq, yv);
    float u[V], ss = 0.f;
#pragma unroll
    for (int v = 0; v < V; ++v) u[v] = 0.f;
#pragma unroll
    for (int t = 0; t < S; ++t) {
        float xt[V];
        if (y) {
#pragma unroll
            for (int v = 0; v < V; ++v) xt[v] = 0.f;
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int v = 0; v < V; ++v) xt[v] += mix[s][t] * xs[s][v];
#pragma unroll
            for (int v = 0; v < V; ++v) xt[v] += to[t] * yv[v];
            if (a.x_out && live) Vec<V>::st(a.x_out + ((long)m * S + t) * H + i, xt);
        } else {
#pragma unroll
            for (int v = 0; v < V; ++v) xt[v] = xs[t][v];
        }
#pragma unroll
        for (int v = 0; v < V; ++v) u[v] += from[t] * xt[v];
    }
    if (a.u_out && live) Vec<V>::st(a.u_out + (long)m * H + i, u);
    if (!normed) return;
#pragma unroll
    for (int v = 0; v < V; ++v) ss = __builtin_fmaf(u[v], u[v], ss);  // (with a choice in the sum it would be a product and an addition: other bits than the loop's)
    const float inv = 1.0f / sqrtf(block_sum(live ? ss : 0.f, red, waves) / (float)H + a.eps);
    if (!live) return;
    float n[V], h[V];
#pragma unroll
    for (int v = 0; v < V; ++v) h[v] = n[v] = u[v] * inv * (a.offset + w[v]);
    if (a.n_out) Vec<V>::st(a.n_out + (long)m * H + i, n);
    if (!a.h) return;
    if (conv) {
        float acc[V];
#pragma unroll
        for (int v = 0; v < V; ++v) acc[v] = 0.f;
#pragma unroll
        for (int k = 0; k < ONCE_TAPS; ++k) {
            if (k + 1 < K) {
#pragma unroll
                for (int v = 0; v < V; ++v) acc[v] += taps[k][v] * before[k][v];
                if (k > 0) Vec<V>::st(tl + (long)(k - 1) * H + i, before[k]);  // each input moves one place towards the oldest
            }
            if (k + 1 == K) {
#pragma unroll
                for (int v = 0; v < V; ++v) h[v] += acc[v] + taps[k][v] * n[v];
            }
        }
        if (K > 1) Vec<V>::st(tl + (long)(K - 2) * H + i, n);
    }
    Vec<V>::st((T*)a.h + (long)m * H + i, h);
}

template <typename T, int S>
static int hyper_launch_s(const HyperArgs& a, int M, bool wide, hipStream_t s) {
    const int per = wide ? 4 : 1;
    const dim3 block(std::min(1024, std::max(64, ((a.H + per - 1) / per + 63) / 64 * 64)));
    const size_t lds = (size_t)a.H * sizeof(float);
    const bool near = a.x_row <= 0xffffffffL && a.x_stream <= 0xffffffffL && a.y_ld <= 0xffffffffL;
    if (near && a.H <= per * (int)block.x && (!a.conv || a.K <= ONCE_TAPS)) {
        const uint32_t sizes = (uint32_t)a.H | (uint32_t)(a.conv ? a.K : 0) << 16 | (a.rows ? 1u << 31 : 0u);
        hipLaunchKernelGGL((wide ? hyper_norm_once_kernel<T, S, 4> : hyper_norm_once_kernel<T, S, 1>), dim3(M), block, 0, s, a.x, (const T*)a.y,
                           a.h || a.n_out ? a.w : nullptr, a.conv, a.token_seq, (uint32_t)a.x_row, (uint32_t)a.x_stream, (uint32_t)a.y_ld, sizes, a.seq_slot, a.mix, a.out, a.in,
                           a.rows, a);
        return pta_check_launch("hyper_norm");
    }
    if (wide) hipLaunchKernelGGL((hyper_norm_kernel<T, S, 4>), dim3(M), block, lds, s, a);
    else hipLaunchKernelGGL((hyper_norm_kernel<T, S, 1>), dim3(M), block, lds, s, a);
    return pta_check_launch("hyper_norm");
}

template <typename T>
static int hyper_launch(const HyperArgs& a, int M, int S, bool wide, hipStream_t s) {
    switch (S) {
        case 1: return hyper_launch_s<T, 1>(a, M, wide, s);
        case 2: return hyper_launch_s<T, 2>(a, M, wide, s);
        case 3: return hyper_launch_s<T, 3>(a, M, wide, s);
        case 4: return hyper_launch_s<T, 4>(a, M, wide, s);
        case 5: return hyper_launch_s<T, 5>(a, M, wide, s);
        case 6: return hyper_launch_s<T, 6>(a, M, wide, s);
        case 7: return hyper_launch_s<T, 7>(a, M, wide, s);
        default: return hyper_launch_s<T, 8>(a, M, wide, s);
    }
}

extern "C" int pta_hyper_norm(void* h, float* n_out, float* u_out, float* x_out, const float* x, long x_row, long x_stream,
                              const void* y, long y_ld, const float* mix, const float* out, const float* in, const float* w,
                              float offset, float eps, const int* rows, const float* conv, int taps, float* tail, long tail_ld,
                              const int* token_seq, const int* seq_slot, int M, int H, int streams, int dtype, void* stream) {
    PTA_REQUIRE(M > 0 && H > 0, "hyper_norm: M=%d H=%d must be positive", M, H);
    PTA_REQUIRE(streams >= 1 && streams <= HYPER_MAX_STREAMS, "hyper_norm: %d streams are outside 1..%d", streams, HYPER_MAX_STREAMS);
    PTA_REQUIRE(H <= 16384, "hyper_norm: rows of %d features are more than the 16384 that fit the kernel's LDS", H);
    PTA_REQUIRE(x && (h || n_out || u_out || x_out), "hyper_norm: null pointer");
    PTA_REQUIRE((h == nullptr && n_out == nullptr) || w, "hyper_norm: a norm needs its weight");
    PTA_REQUIRE(!y || (mix && out && y_ld >= H), "hyper_norm: a sublayer's result needs the streams' mix and its weights");
    PTA_REQUIRE(x_stream == 0 || x_stream >= H, "hyper_norm: streams of %d features cannot lie %ld apart", H, x_stream);
    PTA_REQUIRE(x_row >= (x_stream ? (streams - 1) * x_stream + H : (long)H), "hyper_norm: a token's streams do not fit its row");
    PTA_REQUIRE(!x_out || (y && x_out != x && !rows), "hyper_norm: new streams need a sublayer's result and a buffer of their own");
    PTA_REQUIRE(!conv || (h && taps >= 1 && !rows && token_seq && seq_slot && (taps == 1 || (tail && tail_ld >= (long)(taps - 1) * H))),
                "hyper_norm: the convolution needs its inputs from before the step");
    PTA_REQUIRE(dtype == PTA_F32 || dtype == PTA_BF16, "hyper_norm: unknown dtype %d", dtype);
    const HyperArgs a{h, n_out, u_out, x_out, x, x_row, x_stream, y, y_ld, mix, out, in, w, offset, eps, rows, conv, taps, tail,
                      tail_ld, token_seq, seq_slot, H};
    auto at16 = [](const void* p) { return ((uintptr_t)p % 16) == 0; };
    const bool wide = H % 4 == 0 && x_row % 4 == 0 && x_stream % 4 == 0 && y_ld % 4 == 0 && tail_ld % 4 == 0 && at16(h) && at16(n_out) &&
                      at16(u_out) && at16(x_out) && at16(x) && at16(y) && at16(w) && at16(conv) && at16(tail);
    if (dtype == PTA_F32) return hyper_launch<float>(a, M, streams, wide, (hipStream_t)stream);
    return hyper_launch<bf16_t>(a, M, streams, wide, (hipStream_t)stream);
}
