// The decode-batch product's workgroup (gemm_splitk_bf16.hip says how it works), for its own launch and for the launch that carries a
// decode step's attention as well (gemm_splitk_attn.hip).
#pragma once

#include "common.h"
#include "lds_stream.h"
#include "pta_kernels.h"

// bytes of a stage of 64 elements of K in LDS: the waves' rows of W, and the rows of x by whole loads of each wave (NW: waves, an even number)
static constexpr __host__ __device__ int splitk_slot(int MT, int RT, int NW) { return NW * RT * 2048 + (2 * MT + NW - 1) / NW * NW * 1024; }

#define SK_WAVES 4
#define SK_SIX 6  // waves of a workgroup that has 96 rows of W
#define SK_CHUNK_ROWS 128  // eight tiles of sixteen rows of x: what a workgroup holds
#define SK_MAX_ROWS 256

// One product of a launch.  A launch may carry two that share M (a block's two output projections, left
// as partial sums): the workgroups of the second follow those of the first in a one-dimensional grid.
struct SplitkProblem {
    void* y;
    float* part;
    const bf16_t* x;
    const bf16_t* W;
    const float* bias;
    const bf16_t* add1;
    const bf16_t* add2;
    int N, K, act, out_f32;
    int blocks_per_part;  // 64-element blocks of K per range
    int tiles;            // workgroups along N
    int parts;            // ranges of K
    int direct;           // one range and the epilogue in this kernel
};

// what follows a whole sum, for one element
__device__ __forceinline__ void store_whole(void* y, const float* bias, const bf16_t* add1, const bf16_t* add2, int act, int out_f32, int n,
                                            long o, float v) {
    if (!out_f32) v = round_to_bf16(v);
    if (bias) { v += bias[n]; if (!out_f32) v = round_to_bf16(v); }
    if (act == PTA_ACT_GELU) v = out_f32 ? gelu_erf(v) : gelu_bf16(v);  // other activations: see pta_gemm_splitk_bf16
    if (add1) v += bf16_bits_to_f32(add1[o]);
    if (add2) v += bf16_bits_to_f32(add2[o]);
    if (out_f32) ((float*)y)[o] = v;
    else ((bf16_t*)y)[o] = f32_to_bf16_bits(v);
}

// a launch whose x is there when it starts
struct NoGate {
    static constexpr bool closed = false;
    __device__ __forceinline__ bool wait(bool) const { return true; }
};

// Workgroup `block` of `blocks`.  With a gate that may be closed, x is asked for once the gate is open, and W of the first stages before
// that; false where the gate has used LDS meanwhile and the workgroup is to be begun again.
template <int MT, int RT, int D, bool ROT, int NW, typename Gate>
__device__ __forceinline__ bool splitk_body(const SplitkProblem& pa, const SplitkProblem& pb, int M, int chunks, int chunk_rows,
                                            int rot_stride, int block, int blocks, const Gate& gate) {
    constexpr int NX = (2 * MT + NW - 1) / NW;       // loads of x per wave and stage (eight rows by 128 bytes each)
    constexpr int NL = 2 * RT + NX;                  // all of a wave's loads per stage
    constexpr int SLOT = splitk_slot(MT, RT, NW);    // a stage in LDS: the waves' rows of W, then x
    static_assert(NW % 2 == 0, "a wave's loads of x are all the same half of a tile");
    extern __shared__ __attribute__((aligned(1024))) char lds[];  // [D][SLOT]

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    // More rows than a workgroup holds are cut into `chunks` chunks of `chunk_rows`; the workgroups that take the
    // same rows of W for the chunks sit a multiple of eight apart in the grid, so that they start together on one
    // die and all but the first find W in its cache.
    const int first_blocks = pa.tiles * pa.parts;
    int chunk = 0;
    if (chunks > 1) {
        const int per_chunk = blocks / chunks, whole = per_chunk / 8 * 8, rest = per_chunk - whole;
        if (block < whole * chunks) {
            chunk = (block >> 3) % chunks;
            block = block / (8 * chunks) * 8 + (block & 7);
        } else {
            const int t = block - whole * chunks;
            chunk = t / rest;
            block = whole + t % rest;
        }
    }
    const int m0 = chunk * chunk_rows, m_end = min(M, m0 + chunk_rows);
    const bool second = block >= first_blocks;
    void* __restrict__ y = second ? pb.y : pa.y;
    float* __restrict__ part = second ? pb.part : pa.part;
    const bf16_t* __restrict__ x = second ? pb.x : pa.x;
    const bf16_t* __restrict__ W = second ? pb.W : pa.W;
    const float* __restrict__ bias = second ? pb.bias : pa.bias;
    const bf16_t* __restrict__ add1 = second ? pb.add1 : pa.add1;
    const bf16_t* __restrict__ add2 = second ? pb.add2 : pa.add2;
    const int N = second ? pb.N : pa.N, K = second ? pb.K : pa.K, act = second ? pb.act : pa.act;
    const int out_f32 = second ? pb.out_f32 : pa.out_f32, direct = second ? pb.direct : pa.direct;
    const int blocks_per_part = second ? pb.blocks_per_part : pa.blocks_per_part;
    const int tiles = second ? pb.tiles : pa.tiles;
    const int idx = block - (second ? first_blocks : 0);
    const int tile = idx % tiles, range = idx / tiles;  // neighbours share a range of K: its x slice stays in L2
    const int n_base = tile * (NW * 16 * RT) + wave * (16 * RT);
    const int nkb = (K + 63) >> 6;
    const int kb0 = range * blocks_per_part, kb1 = min(kb0 + blocks_per_part, nkb);
    const int k_begin = kb0 * 64, k_end = min(kb1 * 64, K);
    const int nstages = kb1 - kb0;

    // rows past the last one lie past the buffers' ends, elements past the range's end are asked for there: zeros, no traffic
    const int n_rows = max(0, min(16 * RT, N - n_base));
    const i32x4_t rw = buffer_of(W + (long)min(n_base, N - 1) * K, n_rows * K * 2), rx = buffer_of(x + (long)m0 * K, (m_end - m0) * K * 2);
    const unsigned to_w = __builtin_amdgcn_readfirstlane(lds_address(lds)) + wave * (RT * 2048);
    const unsigned to_x = __builtin_amdgcn_readfirstlane(lds_address(lds)) + NW * RT * 2048 + wave * 1024;
    int w_at[2 * RT], x_at[NX];  // the lane's rows
#pragma unroll
    for (int l = 0; l < 2 * RT; ++l) w_at[l] = ((l >> 1) * 16 + stream_row(lane, l & 1)) * K * 2;
#pragma unroll
    for (int l = 0; l < NX; ++l) {
        const int row = (wave + NW * l) * 8 + (lane >> 3);
        x_at[l] = row < m_end - m0 ? row * K * 2 : LDS_PAST;
    }
    const int c8[2] = {stream_element(lane, 0), stream_element(lane, 1)};

    f32x4_t acc[RT][MT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[t][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // Where a row of W is a power of two long, workgroups that walk the same range of K in step ask the same few
    // memory channels at the same time (N = 4,096, K = 16,384: a third slower than K = 16,448).  So each walks its
    // range from a starting stage of its own and wraps round; stages past the last read nothing.  A feature's
    // order of summation follows from N, K and the launch alone.
    const int rot = ROT && nstages > 0 ? (int)(((long)tile * rot_stride) % nstages) : 0;
    auto k_of = [&](int stage) {
        int at = stage;
        if (ROT) { at += rot; at -= at >= nstages ? nstages : 0; }
        return k_begin + at * 64;
    };
    auto issue_w = [&](int stage, int slot) {
        const int k = k_of(stage);
#pragma unroll
        for (int l = 0; l < 2 * RT; ++l) {
            const int ke = k + c8[l & 1];
            fetch16(rw, to_w + slot + l * 1024, ke < k_end ? w_at[l] + ke * 2 : LDS_PAST);
        }
    };
    auto issue_x = [&](int stage, int slot) {
        const int k = k_of(stage);
#pragma unroll
        for (int l = 0; l < NX; ++l) {
            const int ke = k + c8[wave & 1];  // (an even number of loads away from the wave's first: the same half of a tile)
            fetch16(rx, to_x + slot + l * (NW * 1024), ke < k_end && x_at[l] != LDS_PAST ? x_at[l] + ke * 2 : LDS_PAST);
        }
    };
    auto issue = [&](int stage, int slot) {
        issue_w(stage, slot);
        issue_x(stage, slot);
    };
    const int in_row = r * 128 + ((g ^ (r >> 1)) & 7) * 16;  // the second 32 elements of a stage: 64 flipped
    auto multiply = [&](int cur) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            bf16x8_t w[RT], b[MT];
            const int at = (in_row ^ (hf * 64)) + cur;
#pragma unroll
            for (int t = 0; t < RT; ++t) w[t] = *reinterpret_cast<const bf16x8_t*>(lds + at + (wave * RT + t) * 2048);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) b[mt] = *reinterpret_cast<const bf16x8_t*>(lds + at + NW * RT * 2048 + mt * 2048);
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t], b[mt], acc[t][mt], 0, 0, 0);
        }
    };
    // everyone's share of the stage has landed, and everyone is past reading the one before
    auto meet = [&]() {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // D - 1 stages are on their way, one barrier a stage, behind which the next loads take the place of the stage before; the last
    // D - 1 stages wait for fewer and fewer.
    if constexpr (Gate::closed) {
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < nstages) issue_w(d, d * SLOT);
        if (!gate.wait(second)) return false;
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < nstages) issue_x(d, d * SLOT);
        wait_loads<0>();  // (the loads came in another order than the waits below count)
    } else {
#pragma unroll
        for (int d = 0; d < D - 1; ++d)
            if (d < nstages) issue(d, d * SLOT);
    }
    int cur = 0, free = (D - 1) * SLOT;
    for (int s = D - 1; s < nstages; ++s) {
        wait_reads();
        wait_loads<(D - 2) * NL>();
        meet();
        issue(s, free);
        __builtin_amdgcn_sched_barrier(0);
        multiply(cur);
        free = cur;
        cur = cur == (D - 1) * SLOT ? 0 : cur + SLOT;
    }
    RingTail<NL>::template last_steps<D - 2>(nstages, [&]() {
        meet();
        multiply(cur);
        cur = cur == (D - 1) * SLOT ? 0 : cur + SLOT;
    });

    // lane: row m = mt*16 + r of x, columns n_base + t*16 + g*4 + 0..3
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const int m = m0 + mt * 16 + r, n = n_base + t * 16 + g * 4;
            if (m >= m_end || n >= N) continue;
            const long o = (long)m * N + n;
            if (!direct) {
                const long at = (long)range * M * N + o;
                float* dst = part + at;
                if (n + 3 < N && (at & 3) == 0) *reinterpret_cast<f32x4_t*>(dst) = acc[t][mt];
                else
                    for (int i = 0; i < 4 && n + i < N; ++i) dst[i] = acc[t][mt][i];
                continue;
            }
            for (int i = 0; i < 4 && n + i < N; ++i) store_whole(y, bias, add1, add2, act, out_f32, n + i, o + i, acc[t][mt][i]);
        }
    return true;
}
