// Causal attention over the paged cache on the matrix cores, bfloat16 in, 32-bit softmax and
// accumulation: the prefill kernel and the decode kernel are the same code.
//
// Work is laid out in *columns*: a column is one (new token, query head) pair of one KV head of one
// sequence, ordered token-major.  Heads that share a KV head therefore sit side by side and read
// its keys and values once: with one KV head for 71 query heads, a decode step's 71 columns are five
// tiles of 16 that share every key load.  A wave owns CT column tiles and walks the keys 32 at a
// time, always with the next block's keys and values already on their way:
//
//   S^T[32 keys x 16 cols]  = K[32 x d] . Q^T[d x 16]         (A = key rows, B = query columns)
//   online softmax over keys, per column (statistics in 32-bit, four lanes hold a column)
//   O^T[d x 16 cols]       += V^T[d x 32 keys] . P^T[32 x 16]  (A = value pages, stored transposed)
//   l[16 cols]             += 1[16 x 32] . P^T[32 x 16]        (the sums of the weights, as they were rounded)
//
// The score tile's accumulator layout (lane: column = lane % 16, four consecutive rows at
// (lane / 16) * 4) is turned into the B operand of the second product without leaving registers:
// key rows are assigned to the two 16-row score tiles so that a lane ends up with the eight
// consecutive keys 8 * (lane / 16) .. + 7 of the block, which is what the B operand wants.
//
// Decoding splits a long context over several workgroups (split_size keys each); each writes an
// unnormalised partial result with its running maximum and sum, and attn_combine merges them in split
// order.  A workgroup is one wave, or four or eight that take its keys block by block in turn and merge
// through LDS in the order of the waves; with the whole context in one workgroup there is no second
// launch, but all of a sequence's keys then pass through one compute unit.  Prefill does not split.
//
// `sink` (null: none): a learned number per head whose exponential joins the sum of the weights, once per row, when
// the row's result is normalised (here without ranges of keys, in the merge with them); it has no key and no value.
//
// score = q . k / sqrt(d) + alibi, alibi = bf16(bf16(slope) * bf16(key position)) / sqrt(d)
// (src/transformers/models/falcon/modeling_falcon.py:371-386, :407-422, :196-198, :1078-1085).
#pragma once

#include "common.h"
#include "pta_kernels.h"
#include "score_bias.h"

#include <stddef.h>
#include <stdlib.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

union AFrag {
    uint4 u;
    bf16x8_t v;
};

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// two 32-bit floats to two bfloat16 (round to nearest even) in one instruction
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    union { bf16x2_t b; uint32_t u; } c;
    c.b = __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t);
    return c.u;
}

// The largest of three in one instruction, by the maximum that takes values as they are (fmaxf of values that come through a branch has each made
// canonical by an instruction of its own first).  Not inline asm: the compiler knows nothing of what that reads, and leaves out the wait that a matrix
// instruction's result needs, so scores were read before they were there.  (A NaN stays one: its column's result is NaN in any case.)
// PLAIN: by fmaxf, for the one kernel whose registers the compiler does not come to terms with otherwise.
template <bool PLAIN> __device__ __forceinline__ float max3(float a, float b, float c) {
    if constexpr (PLAIN) return fmaxf(fmaxf(a, b), c);
    else return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}

#define PTA_LOG2E 1.4426950408889634f

template <int DT>
struct KvBlock {
    AFrag k[2][(DT + 1) / 2];
    AFrag v[DT];
};

// Keys and values of the 32-key block at kb, straight into matrix-operand registers.  Nothing here
// depends on the loaded data, so the loads of the next block stay in flight while this one is used.
template <int DT>
__device__ __forceinline__ void load_block(KvBlock<DT>& b, int kb, long page,
                                           const bf16_t* __restrict__ k_pool, const bf16_t* __restrict__ v_pool,
                                           int nkv, int kvh, int c, int gq) {
    constexpr int D = DT * 16, DS = (DT + 1) / 2, CHUNKS = D / 8;
    const int in_page = kb & 63;
    const bf16_t* kpage = k_pool + (page * nkv + kvh) * (long)(PTA_PAGE * D);
    const bf16_t* vpage = v_pool + (page * nkv + kvh) * (long)(PTA_PAGE * D);
    // key rows: tile tt, row r holds key 8*(r/4) + 4*tt + r%4 of the block
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
        const bf16_t* kp = kpage + (long)(in_page + 8 * (c >> 2) + 4 * tt + (c & 3)) * D;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds)
            b.k[tt][ds].u = *reinterpret_cast<const uint4*>(kp + min(ds * 4 + gq, CHUNKS - 1) * 8);
    }
    // value rows: feature dt*16 + c, keys 8*gq .. 8*gq+7 of the block
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        b.v[dt].u = *reinterpret_cast<const uint4*>(vpage + (long)(dt * 16 + c) * PTA_PAGE + in_page + gq * 8);
}

// what the kernel looks at later: read where it is used
struct AttnMore {
    int n_seqs, ranges, split_size, bias_mode, window_arg, chunk_arg;
    float scale, alibi_mul;
    const float* slopes;
    bf16_t* out;
    float *po, *pm, *pl;
    const float* sink;
    PtaHeadRows rows;
};

// A launch's arguments, as the kernel takes them.  What comes first and packed is in registers when a workgroup starts, fourteen words of it: what keys
// and queries are found by.  The others are a load away, which over cold caches takes 0.7 us, and the compiler moves such loads to the front, where the
// first others that are waited for (the block table's, the lengths') are then waited for with them.  So the kernel reads them from where they lie, where it says so.
// With all in its order and asked for at the front, 5 sequences of 40 to 325 keys, 13 heads of 80, took 8.6 us a launch in a step, and take 7.5.
struct AttnKernelArgs {
    const int *block_table, *cu_tokens, *seq_start;
    const bf16_t *k_pool, *v_pool, *q;
    uint32_t heads, table;  // heads of a KV head << 16 | KV heads; pages in a row of the table, and in the two highest bits whether there are ranges and `paired`
    AttnMore more;
};
typedef const __attribute__((address_space(4))) AttnMore& AttnLate;
__device__ __forceinline__ AttnLate attn_late() {
    const __attribute__((address_space(4))) char* at = (const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(at));
    return *(const __attribute__((address_space(4))) AttnMore*)(at + offsetof(AttnKernelArgs, more));
}

// W = 1: a workgroup is one wave, which loads its keys and values straight from global memory.
// W > 1 (prompts; one token per sequence with many heads on a KV head): W waves with neighbouring column groups
// walk the keys together and share every block through LDS, so that a block crosses the vector memory path once
// for 16 * W * CT columns.
// WIN: the launch has a window (a kernel of its own, so that launches without one pay nothing for it).
// KS > 1 (one token per sequence): KS waves of a workgroup hold the same columns and take every KS-th block of the
// workgroup's keys; their partial results meet in LDS, so that a context walked by KS waves needs no second launch.
// AL: whether there is ALiBi, known when the kernel is compiled (0: none, 1: there is) or looked up (2).
// OCC: waves that a SIMD is to hold at least (the registers a wave may use follow from it; 1: as many as it likes).
template <int DT, int CT, int W, bool WIN, int KS = 1, int AL = 2, int OCC = 1>
__global__ __launch_bounds__(64 * W * KS, OCC) void attn_mfma_kernel(
    const int* __restrict__ block_table, const int* __restrict__ cu_tokens, const int* __restrict__ seq_start, const bf16_t* __restrict__ k_pool,
    const bf16_t* __restrict__ v_pool, const bf16_t* __restrict__ q, uint32_t heads, uint32_t table,
    const AttnMore) {  // AttnKernelArgs
    const int g = heads >> 16, nkv = heads & 0xffff, nh = g * nkv, bt_stride = table & 0x3fffffff;
    const bool many_ranges = table >> 31;
    const int paired = KS > 1 ? 0 : table >> 30 & 1;
#define ATTN_X blockIdx.x
#define ATTN_Y blockIdx.y
#define ATTN_Z blockIdx.z
#define ATTN_NX gridDim.x
#define ATTN_INSIDE 0
#define ATTN_LATE(more) AttnLate more = attn_late()
#include "attn_mfma_body.h"
#undef ATTN_X
#undef ATTN_Y
#undef ATTN_Z
#undef ATTN_NX
#undef ATTN_INSIDE
#undef ATTN_LATE
}

struct AttnLaunch {
    bf16_t* out; float *po, *pm, *pl;
    const bf16_t *q, *k_pool, *v_pool;
    const int* block_table; int bt_stride;
    const int *cu_tokens, *seq_start; const float* slopes; int bias_mode; float bias_scale; const float* sink;
    int n_seqs, max_new, nh, nkv; float scale;
    int split_size, n_splits, window;
    int chunk;   // 0, or the size of the blocks of positions that a token does not see out of
    int paired;  // workgroups take two column groups each, a late one and the early one that mirrors it
    int waves;   // one token per sequence: waves of a workgroup that divide its keys among them
    PtaHeadRows rows;
    hipStream_t s;
};

// LDS in which KS waves of CT column tiles leave their partial results
constexpr size_t key_split_lds(int dt, int ct, int ks) { return ks == 1 ? 0 : (size_t)ks * ct * (dt * 1024 + 128); }

template <int DT, int CT, int W, int KS = 1, int OCC = 1>
static void launch_attn(const AttnLaunch& a) {
    const int g = a.nh / a.nkv;
    const int groups = (a.max_new * g + 16 * CT * W - 1) / (16 * CT * W);
    const int paired = a.paired && groups > 1 ? 1 : 0;
    const dim3 grid(paired ? (groups + 1) / 2 : groups, a.nkv, a.n_seqs * a.n_splits);
    // prompts: a kernel with ALiBi and one without; one token per sequence: one kernel that looks
    constexpr int AL0 = W > 1 ? 0 : 2, AL1 = W > 1 ? 1 : 2;
    auto kern = (a.window > 0 || a.chunk > 0) ? attn_mfma_kernel<DT, CT, W, true, KS, AL0, OCC> : attn_mfma_kernel<DT, CT, W, false, KS, AL0, OCC>;
    if (W > 1 && a.slopes)
        kern = (a.window > 0 || a.chunk > 0) ? attn_mfma_kernel<DT, CT, W, true, KS, AL1, OCC> : attn_mfma_kernel<DT, CT, W, false, KS, AL1, OCC>;
    constexpr size_t lds = key_split_lds(DT, CT, KS);
    if constexpr (lds > 64 * 1024) {  // more than a launch may ask for unless the kernel has been told, once per device
        static bool told[64] = {};
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
        if (!told[dev]) {
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            told[dev] = true;
        }
    }
    hipLaunchKernelGGL(kern, grid, dim3(64 * W * KS), lds, a.s, a.block_table, a.cu_tokens, a.seq_start, a.k_pool, a.v_pool, a.q,
                       (uint32_t)g << 16 | (uint32_t)a.nkv, (uint32_t)a.bt_stride | (a.n_splits > 1 ? 1u << 31 : 0u) | (uint32_t)paired << 30,
                       AttnMore{a.n_seqs, a.n_splits, a.split_size, a.bias_mode, a.window, a.chunk, a.scale * PTA_LOG2E, PTA_LOG2E * a.bias_scale, a.slopes,
                                a.out, a.po, a.pm, a.pl, a.sink, a.rows});
}

// column tiles (of sixteen query heads of one KV head) that one wave of a decode launch holds at most:
// what the head size leaves registers for
constexpr int decode_max_tiles(int dt) { return dt <= 4 ? 5 : dt <= 8 ? 4 : 1; }

// waves that may divide a workgroup's keys: one, or four or eight with up to two column tiles each (more tiles
// gained nothing with more waves wherever that was measured, and every combination is a kernel to build)
constexpr bool decode_waves_built(int dt, int ct, int ks) {
    return ks == 1 || ((ks == 4 || ks == 8) && ct <= 2 && ct <= decode_max_tiles(dt) &&
                       key_split_lds(dt, ct, ks) <= 144 * 1024);
}

template <int DT, int CT, int KS = 1>
static bool launch_decode_waves(const AttnLaunch& a) {
    if constexpr (KS <= 8) {
        if (a.waves == KS) {
            if constexpr (decode_waves_built(DT, CT, KS)) { launch_attn<DT, CT, 1, KS>(a); return true; }
            return false;
        }
        return launch_decode_waves<DT, CT, KS * 2>(a);
    }
    return false;
}

// one token per sequence: workgroups of `waves` waves with `tiles` column tiles
template <int DT, int CT = 1>
static bool launch_decode(const AttnLaunch& a, int tiles) {
    if constexpr (CT <= decode_max_tiles(DT)) {
        if (tiles == CT) return launch_decode_waves<DT, CT>(a);
        return launch_decode<DT, CT + 1>(a, tiles);
    }
    return false;
}

// prompts: four waves of two column tiles share each stage of keys through LDS (head sizes up to 128;
// beyond, one wave per workgroup).  Heads up to 64 fit four waves a SIMD (measured at 8,192 tokens, 71 heads
// on one KV head of 64: as many registers as the compiler likes, three waves, 800 us a layer; four waves 760;
// a third column tile, 256 registers, two waves, 817), and with many column groups eight waves share a stage
// (`wide`: 256 columns a workgroup, half the staging for every wave).
constexpr int prompt_columns(int dt, bool wide) { return dt <= 4 && wide ? 256 : dt <= 8 ? 128 : 16; }

template <int DT>
static void launch_prompt(const AttnLaunch& a, bool wide) {
    if constexpr (DT <= 4) {
        if (wide) launch_attn<DT, 2, 8, 1, 4>(a);
        else launch_attn<DT, 2, 4, 1, 4>(a);
    } else if constexpr (DT <= 8) launch_attn<DT, 2, 4>(a);
    else launch_attn<DT, 1, 1>(a);
}

// One token per sequence, the heads of a KV head on the waves of one workgroup, which share its keys through LDS
// as a prompt's column groups do: a wave per tile of sixteen heads for four or five tiles (49 to 80 heads on a KV
// head), four waves of two tiles for six to eight.  Built for head sizes 64 and 128.  Fewer heads on a KV head fit
// the tiles of one wave (`launch_decode`), which reads the keys once as well.
constexpr bool decode_shared_built(int dt, int tiles) { return (dt == 4 || dt == 8) && tiles >= 4 && tiles <= 8; }

template <int DT>
static bool launch_decode_shared(const AttnLaunch& a) {
    if constexpr (DT == 4 || DT == 8) {
        constexpr int OCC = DT <= 4 ? 4 : 1;
        const int tiles = (a.nh / a.nkv + 15) / 16;
        if (tiles == 4) launch_attn<DT, 1, 4, 1, OCC>(a);
        else if (tiles == 5) launch_attn<DT, 1, 5, 1, OCC>(a);
        else if (tiles >= 6 && tiles <= 8) launch_attn<DT, 2, 4, 1, OCC>(a);
        else return false;
        return true;
    }
    return false;
}

// What pta_attn_mfma launches for heads of DT x 16 elements.  Every head size is a translation unit of its own
// (attn_mfma_dt*.hip, one explicit instantiation each), so that the sizes compile side by side.
// 0: launched; 1: no kernel with shared keys at this size; 2: no kernel for these waves and column tiles.
template <int DT>
int attn_launch_head(const AttnLaunch& a, bool shared, bool narrow, bool wide, int tiles) {
    if (shared) return launch_decode_shared<DT>(a) ? 0 : 1;
    if (!narrow) {
        launch_prompt<DT>(a, wide);
        return 0;
    }
    return launch_decode<DT>(a, tiles) ? 0 : 2;
}
