// A decode step of the state-space mixer between its two products, one token a sequence, in one launch: the convolution of the token's
// channels with its activation and the convolution's tail moved on, the recurrence (recurrent.hip has both and the arithmetic), and the
// gated RMS norm of every group of heads, out = y silu(z) / sqrt(mean((y silu(z))^2) + eps) * (offset + w).
//
// A workgroup has a group of heads of a sequence, which share B and C and are what the norm's mean is taken over; so every channel, every
// element of the state and every result belongs to one workgroup and nothing is exchanged.  A wave has a head: its lanes take four
// neighbouring columns of the state's 64 and a quarter of its rows, all of them on their way from the start, sixteen bytes a load
// (64 rows by 64 or 128 by 64: 16 or 32 loads a lane), while the convolution is formed.
//
// What bounds it: the state, 32 KB a head read and written, through few compute units (8 a sequence), and a launch's start and end.  8 sequences of 64 heads
// of 64, 8 groups, 128 rows: convolution, tail, recurrence and norm took 26 us as four launches, this 13.8.
#include "common.h"
#include "pta_kernels.h"

#define STEP_P 64          // columns of a head's state
#define STEP_MOST_HEADS 8  // of a group
#define STEP_MOST_TAPS 4

struct SsmStep {
    const float *conv_w, *conv_b;
    float* tail;
    long tail_ld;
    const float *dt_bias, *A_log, *D;
    float* state;
    long state_ld;
    const float* norm_w;
    float offset, eps;
    const int *cu_tokens, *seq_slot;
    int heads, G;
    int four;  // the norm's sum as of rows that are read four elements at a time
};

__device__ __forceinline__ float step_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// dA S + dx b for a lane's row i, as pta_ssm_scan rounds it: every fourth row has the decay's product in the fused operation, the others the input's
__device__ __forceinline__ float moved(int i, float dA, float S, float dx, float b) {
    return i % 4 == 0 ? __builtin_fmaf(dA, S, dx * b) : __builtin_fmaf(dx, b, dA * S);
}

template <typename T, int NPT, int K>
__global__ __launch_bounds__(STEP_MOST_HEADS * 64) void ssm_step_kernel(T* __restrict__ out, const T* __restrict__ proj, long ld, SsmStep a) {
    constexpr int N = 4 * NPT, P = STEP_P, MOST = STEP_MOST_HEADS * P + 2 * N;
    __shared__ __attribute__((aligned(16))) float chan[MOST];  // the group's channels: x of its heads (then what is normed), B, C
    const int s = blockIdx.y, g = blockIdx.x, per = a.heads / a.G;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane >> 4, col = (lane & 15) * 4;
    const int inner = a.heads * P, C = inner + 2 * a.G * N, channels = per * P + 2 * N, h = g * per + wave;
    const T* row = proj + (long)a.cu_tokens[s] * ld;
    const long slot = a.seq_slot[s];
    float* tail = a.tail + slot * a.tail_ld;
    float* sb = a.state + slot * a.state_ld + (long)h * N * P + (long)q * NPT * P + col;
    // the channels that a thread forms: asked for ahead of the state
    constexpr int MINE = (MOST + 63) / 64;  // with one head a group
    constexpr int AHEAD = 2;                // of a thread with seven heads and more
    auto channel = [&](int i) { return i < per * P ? g * per * P + i : i < per * P + N ? inner + g * N + i - per * P : inner + (a.G + g) * N + i - per * P - N; };
    // (as they lie in memory, and a bias from somewhere where there is none: a value widened, or chosen, where it is loaded is waited for
    // there, one channel behind the other and the state behind them all)
    float w[AHEAD][K], old[AHEAD][K - 1], bias[AHEAD];
    T now[AHEAD], z_raw[4];
    const float* biases = a.conv_b ? a.conv_b : a.conv_w;
    auto fetch = [&](int u, int i) {
        const int c = channel(min(i, channels - 1));
        now[u] = row[inner + c];
        bias[u] = biases[c];
#pragma unroll
        for (int k = 0; k < K; ++k) w[u][k] = a.conv_w[(long)c * K + k];
#pragma unroll
        for (int k = 0; k + 1 < K; ++k) old[u][k] = tail[(long)k * C + c];
    };
    auto form = [&](int u, int i) {
        if (i >= channels) return;
        const int c = channel(i);
        float acc = a.conv_b ? bias[u] : 0.f;
        const float x = Io<T>::ld(&now[u]);
#pragma unroll
        for (int k = 0; k + 1 < K; ++k) acc += w[u][k] * old[u][k];
        acc += w[u][K - 1] * x;
        chan[i] = acc / (1.0f + expf(-acc));
#pragma unroll
        for (int k = 0; k + 1 < K; ++k) tail[(long)k * C + c] = k + 2 < K ? old[u][k + 1] : x;
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) fetch(u, threadIdx.x + u * blockDim.x);
    const T dt_raw = row[inner + C + h];
    const float A = a.A_log[h], dt_b = a.dt_bias[h], skip = a.D[h];
    float nw[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        z_raw[e] = row[h * P + col + e];
        nw[e] = a.norm_w[h * P + col + e];
    }
    __builtin_amdgcn_sched_barrier(0);
    float4 S[NPT];
#pragma unroll
    for (int i = 0; i < NPT; ++i) S[i] = *reinterpret_cast<const float4*>(sb + i * P);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) form(u, threadIdx.x + u * blockDim.x);
    for (int j = AHEAD; j < MINE && j * (int)blockDim.x < channels; ++j) {  // groups of few heads
        fetch(0, threadIdx.x + j * blockDim.x);
        form(0, threadIdx.x + j * blockDim.x);
    }
    // the barrier waits for LDS alone: the state stays on its way
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const float dt = step_softplus(Io<T>::ld(&dt_raw) + dt_b), dA = expf(-expf(A) * dt);
    const float4 xv = *reinterpret_cast<const float4*>(chan + wave * P + col);
    const float4 dx = make_float4(dt * xv.x, dt * xv.y, dt * xv.z, dt * xv.w);
    const float4* B = reinterpret_cast<const float4*>(chan + per * P + q * NPT);
    const float4* Cv = reinterpret_cast<const float4*>(chan + per * P + N + q * NPT);
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < NPT; ++i) {
        const float4 b4 = B[i >> 2], c4 = Cv[i >> 2];
        const float b = (i & 3) == 0 ? b4.x : (i & 3) == 1 ? b4.y : (i & 3) == 2 ? b4.z : b4.w;
        const float c = (i & 3) == 0 ? c4.x : (i & 3) == 1 ? c4.y : (i & 3) == 2 ? c4.z : c4.w;
        S[i] = make_float4(moved(i, dA, S[i].x, dx.x, b), moved(i, dA, S[i].y, dx.y, b), moved(i, dA, S[i].z, dx.z, b), moved(i, dA, S[i].w, dx.w, b));
        acc.x += S[i].x * c; acc.y += S[i].y * c; acc.z += S[i].z * c; acc.w += S[i].w * c;
        *reinterpret_cast<float4*>(sb + i * P) = S[i];
    }
    const float y[4] = {column_sum(acc.x) + skip * xv.x, column_sum(acc.y) + skip * xv.y, column_sum(acc.z) + skip * xv.z, column_sum(acc.w) + skip * xv.w};
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float z = Io<T>::ld(&z_raw[e]);
        v[e] = y[e] * (z / (1.0f + expf(-z)));
    }
    if (q == 0) *reinterpret_cast<float4*>(chan + wave * P + col) = make_float4(v[0], v[1], v[2], v[3]);  // (x there was this wave's alone)
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    // Every wave forms the group's sum of squares, in the order in which pta_rmsnorm does: its threads have four neighbours each, or one element and
    // the one 256 further on, its waves' sums are added in turn.
    float ss = 0.f;
    if (a.four) {
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const float4 u = *reinterpret_cast<const float4*>(chan + 4 * (64 * w + lane));
            ss += wave_sum(__builtin_fmaf(u.x, u.x, u.y * u.y) + __builtin_fmaf(u.z, u.z, u.w * u.w));
        }
    } else {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const int at = 64 * w + lane;
            const float lo = at < per * P ? chan[at] : 0.f, hi = at + 256 < per * P ? chan[at + 256] : 0.f;
            ss += wave_sum(__builtin_fmaf(lo, lo, hi * hi));
        }
    }
    const float inv = 1.0f / sqrtf(ss / (float)(per * P) + a.eps);
    if (q != 0) return;
    T* to = out + (long)a.cu_tokens[s] * inner + h * P + col;
#pragma unroll
    for (int e = 0; e < 4; ++e) Io<T>::st(to + e, v[e] * inv * (a.offset + nw[e]));
}

extern "C" int pta_ssm_step_ok(int heads, int P, int N, int G, int K) {
    return heads > 0 && G > 0 && heads % G == 0 && heads / G <= STEP_MOST_HEADS && P == STEP_P && (N == 64 || N == 128) && K >= 2 && K <= STEP_MOST_TAPS;
}

// proj [tokens, gate | x | B | C | dt] of rows `ld` apart, out [tokens, heads * 64]; one token a sequence.
extern "C" int pta_ssm_step(void* out, const void* proj, long ld, const float* conv_w, const float* conv_b, float* tail, long tail_ld,
                            const float* dt_bias, const float* A_log, const float* D, float* state, long state_ld, const float* norm_w, float offset,
                            float eps, const int* cu_tokens, const int* seq_slot, int n_seqs, int heads, int N, int G, int K, int dtype, void* stream) {
    PTA_REQUIRE(n_seqs > 0 && n_seqs <= 65535, "ssm_step: %d sequences", n_seqs);
    PTA_REQUIRE(pta_ssm_step_ok(heads, STEP_P, N, G, K), "ssm_step: no launch for %d heads in %d groups, %d rows of state, %d taps", heads, G, N, K);
    PTA_REQUIRE(out && proj && conv_w && tail && dt_bias && A_log && D && state && norm_w && cu_tokens && seq_slot, "ssm_step: null pointer");
    const long C = (long)heads * STEP_P + 2L * G * N;
    PTA_REQUIRE(ld >= (long)heads * STEP_P + C + heads && tail_ld >= (K - 1) * C && state_ld >= (long)heads * N * STEP_P,
                "ssm_step: rows lie closer together than they are long");
    PTA_REQUIRE(((uintptr_t)state % 16) == 0 && state_ld % 4 == 0, "ssm_step: rows of state must be 16-byte aligned");
    PTA_REQUIRE(dtype == PTA_F32 || dtype == PTA_BF16, "ssm_step: unknown dtype %d", dtype);
    // where pta_rmsnorm reads a group of 512 and its gate so
    const int four = heads / G * STEP_P == 512 && ld % 4 == 0 && (uintptr_t)proj % (dtype == PTA_F32 ? 16 : 8) == 0 && (uintptr_t)norm_w % 16 == 0;
    const SsmStep a{conv_w, conv_b, tail, tail_ld, dt_bias, A_log, D, state, state_ld, norm_w, offset, eps, cu_tokens, seq_slot, heads, G, four};
    const dim3 grid(G, n_seqs), block(heads / G * 64);
#define STEP(T, NPT, K_) hipLaunchKernelGGL((ssm_step_kernel<T, NPT, K_>), grid, block, 0, (hipStream_t)stream, (T*)out, (const T*)proj, ld, a)
#define STEP_K(T, NPT) if (K == 2) STEP(T, NPT, 2); else if (K == 3) STEP(T, NPT, 3); else STEP(T, NPT, 4)
#define STEP_N(T) if (N == 64) { STEP_K(T, 16); } else { STEP_K(T, 32); }
    if (dtype == PTA_F32) { STEP_N(float); } else { STEP_N(bf16_t); }
#undef STEP
#undef STEP_K
#undef STEP_N
    return pta_check_launch("ssm_step");
}
