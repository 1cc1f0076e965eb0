// y[M,N] = act(x[M,K] . W[N,K]^T + bias) + add1 + add2 for a decode batch of up to 128 rows,
// bfloat16 in, 32-bit accumulation on the matrix cores.
//
// With more than 16 rows the activations are no longer negligible beside the weights: a wave that
// fetched its own x fragments would pull as many bytes of x out of L2 as of W out of HBM.  Here a
// workgroup of four waves owns 64*RT rows of W (16*RT each) and a range of K, and shares x: a stage is 64
// elements of K, for which each wave brings its own rows of W and its share of the rows of x straight to LDS
// (lds_stream.h), D - 1 stages ahead, with one barrier a stage.  K is split over gridDim.y workgroups when N alone
// gives too few of them to occupy the chip; each writes its 32-bit partial tile to `part`, and a second small kernel
// adds the partials in the order of the ranges and applies bias, activation and additions; with reduce = 0 the partials
// are the result, and the kernel that reads them next adds them in the same order.  The split of a product on its own is chosen
// from N and K alone, so its order of summation does not depend on the batch; pairs have one for steps of up to 32 rows, one for
// 33 to 64 and one for more.
//
// Through registers, sixteen rows of W a load, the same ranges took (pairs of products, us, registers -> LDS): 4,544 x 4,544 with
// 4,544 x 18,176 1 row 42.7 -> 40.5, 32 rows 49.6 -> 45.0; 4,096 x 4,096 with 4,096 x 16,384 39.8 -> 36.1, 46.0 -> 39.3; 9,216 and 32,768 x
// 8,192 17 rows 156 -> 139, 32 rows 166 -> 144.
//
// Chunks of x and W past the workgroup's K range, or rows past M and N, are read through a buffer descriptor at
// an offset outside its bounds and arrive as zeros.
#include "gemm_splitk_attn.h"
#include "qkv_tail.h"

#include <stdlib.h>

#include <algorithm>
#include <array>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

template <int MT, int RT, int D, bool ROT, int NW>
__global__ __launch_bounds__(NW * 64) void gemm_splitk_kernel(SplitkProblem pa, SplitkProblem pb, int M, int chunks,
                                                                 int chunk_rows, int rot_stride) {
    splitk_body<MT, RT, D, ROT, NW>(pa, pb, M, chunks, chunk_rows, rot_stride, (int)blockIdx.x, (int)gridDim.x, NoGate{});
}

// The same sums for rows too long for 32-bit offsets within a wave's rows of W (32 rows of 2^25 elements, 16 of 2^26), at most 31 of x: a
// wave takes a row of W by a range of K, four rows of x at a time.
__global__ __launch_bounds__(64) void gemm_splitk_long_kernel(SplitkProblem p, int M) {
    const int lane = threadIdx.x, n = blockIdx.x, range = blockIdx.y;
    const long k0 = (long)range * p.blocks_per_part * 64, k1 = min((long)p.K, k0 + (long)p.blocks_per_part * 64);
    for (int m0 = 0; m0 < M; m0 += 4) {
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        for (long k = k0 + lane * 8; k < k1; k += 512) {  // K is a multiple of 8
            float w[8];
            unpack8(*reinterpret_cast<const uint4*>(p.W + (long)n * p.K + k), w);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float x[8];
                unpack8(*reinterpret_cast<const uint4*>(p.x + (long)min(m0 + i, M - 1) * p.K + k), x);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[i] += x[e] * w[e];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[i] = wave_sum(v[i]);
            if (lane != 0 || m0 + i >= M) continue;
            const long o = (long)(m0 + i) * p.N + n;
            if (p.direct) store_whole(p.y, p.bias, p.add1, p.add2, p.act, p.out_f32, n, o, v[i]);
            else p.part[(long)range * M * p.N + o] = v[i];
        }
    }
}

// y = act(sum over the parts + bias) + add1 + add2; parts are added in the order of their K ranges
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(void* __restrict__ y, const float* __restrict__ part,
                                                                 const float* __restrict__ bias,
                                                                 const bf16_t* __restrict__ add1,
                                                                 const bf16_t* __restrict__ add2, long MN, int N,
                                                                 int P, int act, int out_f32) {
    const long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= MN) return;
    float v = part[o];
    for (int p = 1; p < P; ++p) v += part[(long)p * MN + o];
    const int n = (int)(o % N);
    if (!out_f32) v = round_to_bf16(v);
    if (bias) { v += bias[n]; if (!out_f32) v = round_to_bf16(v); }
    if (act) v = out_f32 ? apply_act(v, act) : apply_act_bf16(v, act);
    if (add1) v += bf16_bits_to_f32(add1[o]);
    if (add2) v += bf16_bits_to_f32(add2[o]);
    if (out_f32) ((float*)y)[o] = v;
    else ((bf16_t*)y)[o] = f32_to_bf16_bits(v);
}

// the same for the two products of a pair launch, bfloat16 out, no additions
__global__ __launch_bounds__(256) void gemm_splitk_reduce2_kernel(bf16_t* __restrict__ y1, const float* __restrict__ part1,
                                                                  const float* __restrict__ bias1, long MN1, int N1, int P1,
                                                                  int act1, bf16_t* __restrict__ y2,
                                                                  const float* __restrict__ part2,
                                                                  const float* __restrict__ bias2, long MN2, int N2, int P2,
                                                                  int act2) {
    long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const bool second = o >= MN1;
    if (second) o -= MN1;
    const long MN = second ? MN2 : MN1;
    if (o >= MN) return;
    const float* part = second ? part2 : part1;
    const float* bias = second ? bias2 : bias1;
    const int N = second ? N2 : N1, P = second ? P2 : P1, act = second ? act2 : act1;
    float v = part[o];
    for (int p = 1; p < P; ++p) v += part[(long)p * MN + o];
    v = round_to_bf16(v);
    if (bias) v = round_to_bf16(v + bias[(int)(o % N)]);
    if (act) v = apply_act_bf16(v, act);
    (second ? y2 : y1)[o] = f32_to_bf16_bits(v);
}

// The reduction on its own, for partial sums that something else made (the vendor library's batched product
// over ranges of K): y[M, N] = act(sum over part[P, M, N] in order + bias) + add1 + add2.
extern "C" int pta_gemm_reduce_parts(void* y, const float* part, const float* bias, const void* add1, const void* add2,
                                     int M, int N, int P, int act, int out_f32, void* stream) {
    PTA_REQUIRE(M > 0 && N > 0 && P > 0, "gemm_reduce_parts: sizes must be positive (M=%d N=%d P=%d)", M, N, P);
    PTA_REQUIRE(y && part, "gemm_reduce_parts: null pointer");
    PTA_REQUIRE(pta_act_known(act), "gemm_reduce_parts: unknown activation %d", act);
    const long MN = (long)M * N;
    PTA_REQUIRE((MN + 255) / 256 < (1L << 31), "gemm_reduce_parts: too many elements for one launch");
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((unsigned)((MN + 255) / 256)), dim3(256), 0, (hipStream_t)stream, y,
                       part, bias, (const bf16_t*)add1, (const bf16_t*)add2, MN, N, P, act, out_f32);
    return pta_check_launch("gemm_reduce_parts");
}

// The reduction of a pair launch whose first product is a fused query_key_value projection: a thread adds the
// partial sums of one pair of a segment's elements (the two that are rotated together, or two that pass;
// qkv_tail_pair_elements) and takes it to its end (qkv_tail.h); the second product as in gemm_splitk_reduce2_kernel, V elements
// a thread (64 rows of 18,176 beside 4,672, one at a time: 5,100 workgroups and 5.9 us; four: 5.5).
template <int V>
__global__ __launch_bounds__(256) void gemm_splitk_reduce2_qkv_kernel(QkvTail tail, const float* __restrict__ part1,
                                                                      const float* __restrict__ bias1, long MN1, int N1,
                                                                      int P1, bf16_t* __restrict__ y2,
                                                                      const float* __restrict__ part2,
                                                                      const float* __restrict__ bias2, long MN2, int N2,
                                                                      int P2, int act2) {
    long o = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long pairs = MN1 >> 1;
    if (o < pairs) {
        const int half = tail.d >> 1, per_row = N1 >> 1;
        const int m = (int)(o / per_row), p = (int)(o % per_row), seg = p / half, i = p % half;
        int ea, eb;
        bool rotated;
        qkv_tail_pair_elements(tail.rot, tail.d, i, ea, eb, rotated);
        const long lo = (long)m * N1 + (long)seg * tail.d + ea, hi = (long)m * N1 + (long)seg * tail.d + eb;
        float a = part1[lo], b = part1[hi];
        for (int q = 1; q < P1; ++q) { a += part1[(long)q * MN1 + lo]; b += part1[(long)q * MN1 + hi]; }
        qkv_tail_pair(tail, bias1, m, seg, i, round_to_bf16(a), round_to_bf16(b));
        return;
    }
    o = (o - pairs) * V;
    if (o >= MN2) return;
    float v[V];
    auto part_at = [&](int q, float (&to)[V]) {
        const float* from = part2 + (long)q * MN2 + o;
        if constexpr (V == 4) *reinterpret_cast<float4*>(to) = *reinterpret_cast<const float4*>(from);
        else to[0] = *from;
    };
    part_at(0, v);
    for (int q = 1; q < P2; ++q) {
        float more[V];
        part_at(q, more);
#pragma unroll
        for (int e = 0; e < V; ++e) v[e] += more[e];
    }
    const int n = bias2 ? (int)(o % N2) : 0;
    bf16_t y[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
        v[e] = round_to_bf16(v[e]);
        if (bias2) v[e] = round_to_bf16(v[e] + bias2[n + e]);
        if (act2) v[e] = apply_act_bf16(v[e], act2);
        y[e] = f32_to_bf16_bits(v[e]);
    }
    if constexpr (V == 4) *reinterpret_cast<uint2*>(y2 + o) = make_uint2((uint32_t)y[0] | (uint32_t)y[1] << 16, (uint32_t)y[2] | (uint32_t)y[3] << 16);
    else y2[o] = y[0];
}

static int pick_rt(int N) { return N >= 16384 ? 2 : 1; }

// ranges that are not empty when K is cut into `parts` ranges of whole 64-element blocks
static int effective_parts(int K, int parts) {
    const int nkb = (K + 63) / 64, per = (nkb + parts - 1) / parts;
    return (nkb + per - 1) / per;
}

// Ranges of K (workgroups along gridDim.y).  Measured at K = 4,096 to 32,768 and N = 4,096 to 32,768: a workgroup does best
// with a range of about 2,304 elements (some 290 KB of weights for its 64 rows), and a launch with at least
// some 512 workgroups; no range is shorter than 512 elements, and there are at most 16.
#define SK_RANGE 2304
static int splitk_target() {
    static const int target = getenv("PTA_SPLITK_WGS") ? atoi(getenv("PTA_SPLITK_WGS")) : 512;
    return target;
}
static int clamp_parts(int P, int K) { return max(1, min(min(P, 16), max(1, K / 512))); }

// with many row tiles the ranges may be longer: fewer partial sums for the same number of workgroups
static int range_for(int groups) { return SK_RANGE * max(1, groups / 64); }

// Among the counts near that rule's, the one with the least (rounds of workgroups on the chip's compute units)
// x (a workgroup's fixed cost + the length of its range).  Measured at 32 to 128 rows: a launch just over a whole
// number of rounds pays for the last one in full (N = 9,216 and K = 8,192, 144 row tiles: 4 ranges, 2.25 rounds, 81
// us; 3 ranges, 1.69 rounds, 65 us; N = 4,672 and K = 4,544, 73 row tiles: 8 ranges 31.6 us, 7 ranges 27.6 us), and the fixed
// cost of a workgroup (start, first loads, its tile of partial sums) is that of some 1,300 elements of K.
#define SK_WG_FIXED 1300
static int pick_parts(int N, int K, int rt) {
    const int groups = (N + 64 * rt - 1) / (64 * rt), range = range_for(groups);
    const int p0 = clamp_parts(max((splitk_target() + groups - 1) / groups, (K + range / 2) / range), K);
    const long units = max(1, pta_compute_units());
    auto cost = [&](int p) { return (((long)groups * p + units - 1) / units) * (SK_WG_FIXED + K / p); };
    static const bool balance = !getenv("PTA_SPLITK_BALANCE") || atoi(getenv("PTA_SPLITK_BALANCE")) != 0;
    int best = p0;
    for (int p = max(1, p0 - 2); balance && p <= p0 + 2; ++p) {
        if (clamp_parts(p, K) != p || effective_parts(K, p) != p || (long)groups * p < 384) continue;
        if (cost(p) < cost(best)) best = p;
    }
    return best;
}

extern "C" int pta_gemm_splitk_parts(int N, int K, int parts, int rt) {
    if (N <= 0 || K <= 0) return 0;
    if (rt <= 0) rt = pick_rt(N);
    return effective_parts(K, parts > 0 ? parts : pick_parts(N, K, rt));
}

// How a pair runs: 1 or 2, workgroups of four waves with so many tiles of sixteen rows of W each; 3, with stationary activations; 4, of six waves with
// a tile each.
#define PAIR_STATIONARY 3
#define PAIR_SIX 4
static int tile_rows(int kind) { return kind == PAIR_SIX ? 16 * SK_SIX : 64 * kind; }  // of W, of a workgroup

static SplitkProblem make_problem(void* y, float* part, const void* x, const void* W, const float* bias,
                                  const void* add1, const void* add2, int N, int K, int act, int out_f32, int rt,
                                  int parts, int reduce) {
    SplitkProblem p{};
    p.y = y; p.part = part; p.x = (const bf16_t*)x; p.W = (const bf16_t*)W; p.bias = bias;
    p.add1 = (const bf16_t*)add1; p.add2 = (const bf16_t*)add2;
    p.N = N; p.K = K; p.act = act; p.out_f32 = out_f32;
    const int nkb = (K + 63) / 64;
    p.blocks_per_part = (nkb + parts - 1) / parts;
    p.parts = (nkb + p.blocks_per_part - 1) / p.blocks_per_part;  // ranges that are not empty
    p.tiles = (N + tile_rows(rt) - 1) / tile_rows(rt);
    p.direct = reduce && p.parts == 1;
    return p;
}

static int reduce_parts(const SplitkProblem& a, int M, int reduce, hipStream_t s) {
    if (reduce && a.parts > 1) {
        const long MN = (long)M * a.N;
        hipLaunchKernelGGL(gemm_splitk_reduce_kernel, dim3((unsigned)((MN + 255) / 256)), dim3(256), 0, s, a.y, a.part,
                           a.bias, a.add1, a.add2, MN, a.N, a.parts, a.act, a.out_f32);
    }
    return pta_check_launch("gemm_splitk_bf16");
}

// rows of W a multiple of 4 KB long are the ones that crowd memory channels: there every workgroup starts at a
// stage of its own (PTA_SPLITK_ROT: stages between neighbours, 0 switches it off)
static int rotation_stride() {
    static const int env = getenv("PTA_SPLITK_ROT") ? atoi(getenv("PTA_SPLITK_ROT")) : -1;
    return env >= 0 ? env : 1;
}
static bool crowding(int K) { return rotation_stride() > 0 && K % 2048 == 0; }
static bool rotated(const SplitkProblem& a, const SplitkProblem& b) { return crowding(a.K) || (b.N > 0 && crowding(b.K)); }

// (x lies within 32-bit offsets: check_splitk)
static bool rows_too_long(const SplitkProblem& a, const SplitkProblem& b, int rt) { return (long)std::max(a.K, b.K) * 16 * rt * 2 >= LDS_PAST; }

template <int MT, int RT, int NW = SK_WAVES>
static int launch_cfg(const SplitkProblem& a, const SplitkProblem& b, int M, int reduce, hipStream_t s) {
    constexpr int D = 4;  // stages in LDS
    constexpr int lds = D * splitk_slot(MT, RT, NW);
    static_assert(lds <= 160 * 1024, "the stages must fit the LDS of a compute unit");
    const int rot_stride = rotation_stride();
    const bool rotate = rotated(a, b);
    auto kern = rotate ? gemm_splitk_kernel<MT, RT, D, true, NW> : gemm_splitk_kernel<MT, RT, D, false, NW>;
    if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return pta_fail("gemm_splitk_bf16: cannot have %d bytes of LDS", lds);
    if (rows_too_long(a, b, RT)) {
        for (const SplitkProblem* p : {&a, &b})
            if (p->N > 0) hipLaunchKernelGGL(gemm_splitk_long_kernel, dim3(p->N, p->parts), dim3(64), 0, s, *p, M);
        return reduce_parts(a, M, reduce, s);
    }
    // rows beyond the MT tiles of a workgroup go to further chunks of workgroups, all of the same size
    const int chunks = (M + MT * 16 - 1) / (MT * 16), chunk_rows = ((M + chunks - 1) / chunks + 15) / 16 * 16;
    const dim3 grid((a.tiles * a.parts + b.tiles * b.parts) * chunks);
    hipLaunchKernelGGL(kern, grid, dim3(NW * 64), lds, s, a, b, M, chunks, chunk_rows, rot_stride);
    return reduce_parts(a, M, reduce, s);
}

// sixteen-row tiles of x that a workgroup holds: all rows up to SK_CHUNK_ROWS, else an even share of them
static int tiles_per_chunk(int M) {
    const int chunks = (M + SK_CHUNK_ROWS - 1) / SK_CHUNK_ROWS;
    return ((M + chunks - 1) / chunks + 15) / 16;
}

template <int RT>
static int launch_rows(int MT, const SplitkProblem& a, const SplitkProblem& b, int M, int reduce, hipStream_t s) {
    switch (MT) {
        case 1: return launch_cfg<1, RT>(a, b, M, reduce, s);
        case 2: return launch_cfg<2, RT>(a, b, M, reduce, s);
        case 3: return launch_cfg<3, RT>(a, b, M, reduce, s);
        case 4: return launch_cfg<4, RT>(a, b, M, reduce, s);
        case 5: case 6: return launch_cfg<6, RT>(a, b, M, reduce, s);
        default: return launch_cfg<8, RT>(a, b, M, reduce, s);
    }
}

static int check_splitk(const char* what, const void* x, const void* W, int M, int N, int K) {
    PTA_REQUIRE(M > 0 && N > 0 && K > 0, "%s: sizes must be positive (M=%d N=%d K=%d)", what, M, N, K);
    PTA_REQUIRE(M <= SK_MAX_ROWS, "%s: at most %d rows, got %d (use the library product)", what, SK_MAX_ROWS, M);
    PTA_REQUIRE(K % 8 == 0 && K >= 8, "%s: K=%d must be a multiple of 8 (16-byte loads)", what, K);
    PTA_REQUIRE(x && W, "%s: null pointer", what);
    PTA_REQUIRE((long)M * K * 2 < 0x7ffffff0L, "%s: x is too large for 32-bit buffer offsets", what);
    PTA_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)W % 16) == 0, "%s: x and W must be 16-byte aligned", what);
    return 0;
}

extern "C" int pta_gemm_splitk_bf16(void* y, float* part, const void* x, const void* W, const float* bias,
                                    const void* add1, const void* add2, int M, int N, int K, int act, int out_f32,
                                    int rt, int parts, int stage_blocks, int depth, int reduce, void* stream) {
    if (check_splitk("gemm_splitk_bf16", x, W, M, N, K)) return 1;
    PTA_REQUIRE(y || !reduce, "gemm_splitk_bf16: null pointer");
    PTA_REQUIRE(pta_act_known(act), "gemm_splitk_bf16: unknown activation %d", act);
    PTA_REQUIRE(rt == 0 || rt == 1 || rt == 2, "gemm_splitk_bf16: row tiles per wave must be 0 (choose), 1 or 2, got %d", rt);
    PTA_REQUIRE(stage_blocks == 0 || stage_blocks == 2,
                "gemm_splitk_bf16: 64-element blocks per stage must be 0 (choose) or 2, got %d", stage_blocks);
    PTA_REQUIRE(depth == 0 || depth == 2 || depth == 4, "gemm_splitk_bf16: stages in flight must be 0 (choose), 2 or 4, got %d", depth);
    PTA_REQUIRE(parts >= 0 && parts <= 64, "gemm_splitk_bf16: parts must be 0 (choose) or 1..64, got %d", parts);
    if (rt == 0) rt = pick_rt(N);
    if (parts == 0) parts = pick_parts(N, K, rt);
    SplitkProblem a = make_problem(y, part, x, W, bias, add1, add2, N, K, act, out_f32, rt, parts, reduce);
    PTA_REQUIRE(a.direct || part, "gemm_splitk_bf16: %d ranges of K need the workspace for partial sums", a.parts);
    // One range of K ends in the matrix kernel itself, whose epilogue knows the exact GELU only (every activation
    // there would cost it its unrolled loops): another activation, and the additions after it, run as a pass over y.
    const bool after = a.direct && act != PTA_ACT_NONE && act != PTA_ACT_GELU;
    if (after) {
        PTA_REQUIRE(!out_f32, "gemm_splitk_bf16: activation %d needs a bfloat16 result", act);
        a.act = PTA_ACT_NONE;
        a.add1 = a.add2 = nullptr;
    }
    const SplitkProblem none{};
    hipStream_t s = (hipStream_t)stream;
    const int MT = tiles_per_chunk(M);
    int rc;
    if (rt == 1) rc = launch_rows<1>(MT, a, none, M, reduce, s);
    else rc = launch_rows<2>(MT, a, none, M, reduce, s);
    if (rc || !after) return rc;
    return pta_epilogue(y, N, nullptr, add1, add2, M, N, act, PTA_BF16, stream);
}

// Ranges of K for the two products of a pair launch: each by its own length, and more of both if the launch
// would have too few workgroups.
// Counts that a caller has fixed for the pairs of one shape: no rule tells which neighbour of its choice is the
// fastest (N = 4,096 with K = 4,096 and 16,384 at 64 rows: 2 and 7 ranges by the rule; 4 and 8 make the
// decode step 7 % faster, 2 and 10 make it 3 % slower with as many workgroups), so the Python side times them once.
struct PairChoice { int p1, p2, rt; };
struct PairFixed { PairChoice few, middle; };  // for 33 to 64 rows of wide matrices (staged_middle), and for all others; p1 = 0: the rule's
static std::map<std::array<int, 4>, PairFixed> pair_parts_fixed;
static std::mutex pair_parts_lock;

static bool parts_valid(int K, int p) { return p >= 1 && clamp_parts(p, K) == p && effective_parts(K, p) == p; }

// (At 33 to 64 rows the staged kernel was timed for matrices of 4,096 rows together and more.)
#define STAGED_FROM_ROWS 4096
static bool staged_middle(int N1, int N2) { return N1 + N2 >= STAGED_FROM_ROWS; }

// Fixes, for every later pair launch of this shape, the ranges of K of the two products and how many tiles of
// sixteen rows of W a wave holds in steps of more than 32 rows (rt 1 or 2: 64 or 128 rows of W a workgroup; the
// taller tile loads the activations half as often and has half as many workgroups).  p1 = p2 = 0 forgets the
// shape.  Returns 1 (no error text) for counts that the kernel does not take.  The ranges decide the order of
// summation; the tile height does not.
extern "C" int pta_gemm_splitk_pair_fix(int N1, int K1, int N2, int K2, int p1, int p2, int rt) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0) return 1;
    std::lock_guard<std::mutex> hold(pair_parts_lock);
    const std::array<int, 4> key{N1, K1, N2, K2};
    if (p1 == 0 && p2 == 0) {
        pair_parts_fixed.erase(key);
        return 0;
    }
    if (!parts_valid(K1, p1) || !parts_valid(K2, p2) || (rt != 1 && rt != 2 && rt != PAIR_SIX)) return 1;
    pair_parts_fixed[key] = {{p1, p2, rt}, {p1, p2, rt}};
    return 0;
}

extern "C" int pta_gemm_splitk_pair_fix_parts(int N1, int K1, int N2, int K2, int p1, int p2) {
    return pta_gemm_splitk_pair_fix(N1, K1, N2, K2, p1, p2, 1);
}

// The same for steps of 33 to 64 rows alone, of matrices for which those have ranges of their own (else 1).
extern "C" int pta_gemm_splitk_pair_fix_middle(int N1, int K1, int N2, int K2, int p1, int p2, int rt) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0 || !staged_middle(N1, N2)) return 1;
    if (!parts_valid(K1, p1) || !parts_valid(K2, p2) || (rt != 1 && rt != 2 && rt != PAIR_SIX)) return 1;
    std::lock_guard<std::mutex> hold(pair_parts_lock);
    pair_parts_fixed[{N1, K1, N2, K2}].middle = {p1, p2, rt};  // (a new entry's others are the rule's)
    return 0;
}

// What a pair launch with `a` and `b` ranges takes at so many rows, in microseconds: the workgroups are handed to the compute units in
// turn, as many at a time as LDS has room for (the rest goes to whichever is done first), and the launch takes as long as the unit
// with the most blocks of 64 elements to pull, or as the chip does for all of them; a workgroup starts and ends in the time of six
// blocks, uneven ranges cost 2 %, and partial sums are written and read again.  Put together from 1,500 launches of eight pairs of shapes at 8, 32 and 64
// rows; what it picks takes on average 1 % longer than the fastest of them, at most 5.  Ranges of about 2,304 elements, the rule
// before, and what this picks, us at 8, 32 and 64 rows (64: before with stationary activations):
//   4,544 x 4,544 + 4,544 x 18,176   40.8 -> 40.2   42.9 -> 42.7   48.9 -> 43.9    9,216 + 32,768 x 8,192    129.5 -> 128.0   132.3 -> 129.4   148.6 -> 143.3
//   4,096 x 4,096 + 4,096 x 16,384   36.5 -> 32.9   39.2 -> 33.8   41.4 -> 39.6    8,192 x 8,192 + 32,768    117.9 -> 111.8   127.7 -> 118.4   141.2 -> 139.7
//   2,048 x 2,048 + 2,048 x 8,192    11.2 -> 10.5   12.8 -> 11.1   15.2 -> 13.3    7,680 + 20,480 x 5,120     54.3 -> 52.6    58.6 -> 60.2    71.6 -> 66.3
static double pair_us(int N1, int K1, int a, int N2, int K2, int b, int rt, int rows) {
    const int units = max(1, pta_compute_units()), slots = units * (rt == 1 ? (rows <= 32 ? 3 : 2) : rows <= 16 && rt == 2 ? 2 : 1);
    const double fixed = 6.0;
    struct Run { int count; double blocks; } runs[4];
    int n = 0;
    long groups = 0;
    double total = 0.0, longest = 0.0, uneven = 0.0;
    for (int i = 0; i < 2; ++i) {
        const int N = i ? N2 : N1, K = i ? K2 : K1, p = i ? b : a;
        const int nkb = (K + 63) / 64, per = (nkb + p - 1) / p, parts = (nkb + per - 1) / per, tiles = (N + tile_rows(rt) - 1) / tile_rows(rt);
        runs[n++] = Run{tiles * (parts - 1), per + fixed};
        runs[n++] = Run{tiles, nkb - (parts - 1) * per + fixed};
        groups += (long)tiles * parts;
        if (nkb % parts) uneven += (double)N * K / ((double)N1 * K1 + (double)N2 * K2);
    }
    for (const Run& r : runs) {
        total += r.count * r.blocks;
        if (r.count) longest = std::max(longest, r.blocks);
    }
    std::vector<double> load(units, 0.0);
    int at = 0;
    for (const Run& r : runs)
        for (int j = 0; j < r.count && at < slots; ++j, ++at) load[at % units] += r.blocks;
    const double mean = total / units;
    double most = *std::max_element(load.begin(), load.end());
    if (groups > slots) most = std::max(most, mean + 0.5 * longest);
    const double bytes = 128.0 * tile_rows(rt) + 0.2 * 4096.0 * (((rows + 15) / 16 + 1) / 2);  // of a block: rows of W, and of x, which come from near by
    return 4.0 + (1.0 + 0.02 * uneven) * std::max(most * bytes / 26e3, mean * bytes / 22.5e3) + ((double)a * N1 + (double)b * N2) * rows * 4.0 / 3e6;
}

// Ranges, and tiles of sixteen rows of W a wave, for steps of up to 32 rows (one tile) or of 33 to 64; kept by shape.  96 rows of W on six waves, at 33 to 64
// rows, are for where 64 or 128 leave compute units idle or with twice the rows of others, as a unit pulls some 25 GB/s whatever is on its
// way: 4,672 + 18,176 x 4,544 (179 workgroups of 128 rows, 239 of 96), us at 33 / 48 / 64 rows 41.2 -> 38.7, 43.0 -> 39.4, 45.6 -> 41.5.  They read x more often,
// and are taken where the time says 5 % less: at 4 % less (4,544 x 4,544 + 18,176) they are 2 % the faster at 33 rows and none at 64, at none less (9,216 + 32,768 x
// 8,192) 3 % the slower.  Nor where each tile walks K from a place of its own, which another height of the tiles would change the sums by: 6,144 + 16,384 x 4,096
// took 38.1 -> 37.7, 38.7 -> 38.3, 40.6 -> 39.5, and steps of 40 and 64 rows of eight such layers 22.47 -> 22.33 and 24.65 -> 24.43 ms, no more than runs differ by.
static PairChoice pair_rule(int N1, int K1, int N2, int K2, int rows) {
    static std::map<std::array<int, 5>, PairChoice> known;
    const std::array<int, 5> key{N1, K1, N2, K2, rows};
    std::lock_guard<std::mutex> hold(pair_parts_lock);
    const auto it = known.find(key);
    if (it != known.end()) return it->second;
    PairChoice best{1, 1, 1};
    double us = 1e30;
    for (int rt : {1, 2, PAIR_SIX}) {
        if ((rt > 1 && rows <= 32) || (rt == PAIR_SIX && (crowding(K1) || crowding(K2)))) continue;
        for (int a = 1; a <= 8; ++a)
            for (int b = 1; b <= 16; ++b) {
                if (!parts_valid(K1, a) || !parts_valid(K2, b)) continue;
                const double t = pair_us(N1, K1, a, N2, K2, b, rt, rows);
                if (t < (rt == PAIR_SIX ? 0.95 * us : us)) us = t, best = PairChoice{a, b, rt};
            }
    }
    if (known.size() >= 1024) known.clear();
    return known[key] = best;
}

// the staged kernel's ranges, and its tiles of sixteen rows of W a wave, for a step of so many rows (0: up to 32)
static int pick_pair_parts(int N1, int K1, int N2, int K2, int M, int* p1, int* p2) {
    const bool middle = M > 32 && M <= 64 && staged_middle(N1, N2);
    PairChoice c{0, 0, 1};
    {
        std::lock_guard<std::mutex> hold(pair_parts_lock);
        const auto it = pair_parts_fixed.find({N1, K1, N2, K2});
        if (it != pair_parts_fixed.end()) c = middle ? it->second.middle : it->second.few;
    }
    if (c.p1 == 0) c = pair_rule(N1, K1, N2, K2, middle ? 64 : 32);
    *p1 = c.p1;
    *p2 = c.p2;
    return M <= 32 || (M > 64 && c.rt == PAIR_SIX) ? 1 : c.rt;
}

// Steps of up to 128 rows may run with the activations stationary (gemm_stationary_bf16.hip), which cuts K into
// ranges of its own, by the class of the step's rows (up to 16, 32, 64, 128).  The rule: ranges of about 1,400
// elements, of the same length in both products, but no more of them than leave every wave at most the row tiles
// it can hold with one workgroup per compute unit (past that the launch needs a second round of workgroups).
// Measured against the staged kernel of its time, which brought W to registers (us, staged -> stationary with the rule's ranges): K = 4,544 with N = 4,672
// + 18,176 at 8 / 32 / 64 / 128 rows 45.3 -> 40.5, 47.1 -> 43.1, 58.2 -> 46.5, 75.4 -> 56.0; K = 4,544 + 18,176
// with N = 4,544: 44.9 -> 41.6, 48.8 -> 44.9, 57.5 -> 48.0, 72.6 -> 55.6; K = 4,096 with N = 6,144 + 16,384: 42.3
// -> 38.4, 45.6 -> 40.1, 51.7 -> 45.1, 64.8 -> 55.1; K = 8,192 with N = 9,216 + 32,768: 141.8 -> 137.5, 158.5 ->
// 154.6, 178.9 -> 163.5, 188.7 -> 185.7.  Which count of ranges is fastest varies by a few percent around the
// rule's (and at 128 rows of the last shape three ranges in two rounds beat one by a tenth), so the Python side
// times the neighbours per class and fixes what wins, or the staged kernel where that wins.
#define STATIONARY_MAX_ROWS 128
#define STATIONARY_CLASSES 4
#define STATIONARY_RANGE 1400
static int stationary_class(int M) { return M <= 16 ? 0 : M <= 32 ? 1 : M <= 64 ? 2 : 3; }
struct StationaryChoice { int q1[STATIONARY_CLASSES], q2[STATIONARY_CLASSES]; };  // 0: the staged kernel
static std::map<std::array<int, 4>, StationaryChoice> pair_stationary_fixed;

// Where no choice is fixed the launch is used from 65 rows on: below, the staged kernel is faster (pair_us), at 128 rows 53 us against its
// 57 for 4,672 + 18,176 x 4,544, 163 against 167 for 9,216 + 32,768 x 8,192, 54 against 52 for 4,544 x 4,544 + 4,544 x 18,176, 158 against
// 168 for 8,192 x 8,192 + 32,768.
static bool stationary_unfixed(int N1, int N2, int cls) { return cls >= 3 || (cls == 2 && !staged_middle(N1, N2)); }

static void stationary_rule(int N1, int K1, int N2, int K2, int cls, int* q1, int* q2) {
    const int kmin = min(K1, K2), f1 = max(1, (K1 + kmin / 2) / kmin), f2 = max(1, (K2 + kmin / 2) / kmin);
    const long tiles = (long)((N1 + 15) / 16) * f1 + (long)((N2 + 15) / 16) * f2;
    const long room = (long)pta_compute_units() * 8 * (cls == 3 ? 2 : 3);  // waves x row tiles a wave holds
    int base = max(1, (kmin + STATIONARY_RANGE / 2) / STATIONARY_RANGE);
    base = max(1, (int)min((long)base, room / max(1L, tiles)));
    while (base > 1 && (base * f1 > 16 || base * f2 > 16)) --base;
    *q1 = effective_parts(K1, min(16, base * f1));
    *q2 = effective_parts(K2, min(16, base * f2));
}

// Fixes, for every later pair launch of this shape with rows of class cls (0: up to 16 rows, 1: 32, 2: 64, 3:
// 128), the ranges of K of the launch with stationary activations; q1 = q2 = 0: the staged kernel for the class;
// cls = -1 forgets the shape.  Returns 1 (no error text) for counts that the kernel does not take.
extern "C" int pta_gemm_splitk_pair_fix_stationary(int N1, int K1, int N2, int K2, int cls, int q1, int q2) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0) return 1;
    std::lock_guard<std::mutex> hold(pair_parts_lock);
    const std::array<int, 4> key{N1, K1, N2, K2};
    if (cls == -1) {
        pair_stationary_fixed.erase(key);
        return 0;
    }
    if (cls < 0 || cls >= STATIONARY_CLASSES) return 1;
    const bool staged = q1 == 0 && q2 == 0;
    if (!staged && (q1 < 1 || q2 < 1 || q1 > 16 || q2 > 16 || effective_parts(K1, q1) != q1 || effective_parts(K2, q2) != q2))
        return 1;
    auto it = pair_stationary_fixed.find(key);
    if (it == pair_stationary_fixed.end()) {
        StationaryChoice c{};
        for (int i = 0; i < STATIONARY_CLASSES; ++i)  // the other classes stay as they are
            if (stationary_unfixed(N1, N2, i)) stationary_rule(N1, K1, N2, K2, i, &c.q1[i], &c.q2[i]);
        it = pair_stationary_fixed.emplace(key, c).first;
    }
    it->second.q1[cls] = q1;
    it->second.q2[cls] = q2;
    return 0;
}

// The ranges of a pair launch of M rows and its kind: 3 with stationary activations, else the tiles of sixteen
// rows of W per wave of the staged kernel (1 or 2).  M = 0 asks for the staged kernel's ranges.
static int pick_pair_parts_rows(int N1, int K1, int N2, int K2, int M, int* p1, int* p2) {
    if (M >= 1 && M <= STATIONARY_MAX_ROWS && K1 % 8 == 0 && K2 % 8 == 0) {
        const int cls = stationary_class(M);
        int q1 = 0, q2 = 0;
        bool fixed = false;
        {
            std::lock_guard<std::mutex> hold(pair_parts_lock);
            const auto it = pair_stationary_fixed.find({N1, K1, N2, K2});
            if (it != pair_stationary_fixed.end()) {
                q1 = it->second.q1[cls];
                q2 = it->second.q2[cls];
                fixed = true;
            }
        }
        if (!fixed && stationary_unfixed(N1, N2, cls)) stationary_rule(N1, K1, N2, K2, cls, &q1, &q2);
        if (q1 > 0 && q2 > 0) {
            *p1 = q1;
            *p2 = q2;
            return PAIR_STATIONARY;
        }
    }
    return pick_pair_parts(N1, K1, N2, K2, M, p1, p2);
}

extern "C" int pta_gemm_splitk_pair_parts(int N1, int K1, int N2, int K2, int M, int* p1, int* p2) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0 || M < 0) return pta_fail("gemm_splitk_pair_parts: sizes must be positive");
    pick_pair_parts_rows(N1, K1, N2, K2, M, p1, p2);
    return 0;
}

// The same, and how the launch runs: 1 or 2, tiles of sixteen rows of W a wave of the staged kernel; 3, with stationary activations.
extern "C" int pta_gemm_splitk_pair_way(int N1, int K1, int N2, int K2, int M, int* p1, int* p2, int* way) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0 || M < 0) return pta_fail("gemm_splitk_pair_way: sizes must be positive");
    *way = pick_pair_parts_rows(N1, K1, N2, K2, M, p1, p2);
    return 0;
}

extern "C" int pta_gemm_stationary_rule(int N1, int K1, int N2, int K2, int cls, int* q1, int* q2) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0 || cls < 0 || cls >= STATIONARY_CLASSES)
        return pta_fail("gemm_stationary_rule: sizes must be positive and the class of rows 0 to %d", STATIONARY_CLASSES - 1);
    stationary_rule(N1, K1, N2, K2, cls, q1, q2);
    return 0;
}

// Two products of one launch, both left as partial sums: part1 [parts1, M, N1] of x1 . W1^T and part2
// [parts2, M, N2] of x2 . W2^T, with the ranges pta_gemm_splitk_pair_parts gives for M rows.
extern "C" int pta_gemm_splitk_pair_bf16(float* part1, const void* x1, const void* W1, int N1, int K1, float* part2,
                                         const void* x2, const void* W2, int N2, int K2, int M, void* stream) {
    if (check_splitk("gemm_splitk_pair_bf16", x1, W1, M, N1, K1)) return 1;
    if (check_splitk("gemm_splitk_pair_bf16", x2, W2, M, N2, K2)) return 1;
    PTA_REQUIRE(part1 && part2, "gemm_splitk_pair_bf16: null workspace");
    int p1, p2;
    const int kind = pick_pair_parts_rows(N1, K1, N2, K2, M, &p1, &p2);
    if (kind == PAIR_STATIONARY) return pta_gemm_stationary_pair_bf16(part1, x1, W1, N1, K1, p1, part2, x2, W2, N2, K2, p2, M, stream);
    const SplitkProblem a = make_problem(nullptr, part1, x1, W1, nullptr, nullptr, nullptr, N1, K1, 0, 0, kind, p1, 0);
    const SplitkProblem b = make_problem(nullptr, part2, x2, W2, nullptr, nullptr, nullptr, N2, K2, 0, 0, kind, p2, 0);
    if (kind == PAIR_SIX) return M <= 48 ? launch_cfg<3, 1, SK_SIX>(a, b, M, 0, (hipStream_t)stream) : launch_cfg<4, 1, SK_SIX>(a, b, M, 0, (hipStream_t)stream);
    if (kind == 2) return launch_rows<2>(tiles_per_chunk(M), a, b, M, 0, (hipStream_t)stream);
    return launch_rows<1>(tiles_per_chunk(M), a, b, M, 0, (hipStream_t)stream);
}

// Whether a decode step's attention of so many heads may ride in the launch of a pair: one of the staged kernel's, for steps of up to 64
// rows, heads of 64 elements.
extern "C" int pta_gemm_splitk_pair_attn_ok(int N1, int K1, int N2, int K2, int M, int nh, int nkv, int d) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0 || M <= 0 || M > RIDE_MOST_ROWS || nkv <= 0 || nh <= 0 || nh % nkv || d != 16 * RIDE_HEAD ||
        (long)nh * d != K2 || K1 % 8 || K2 % 8)
        return 0;
    int p1, p2;
    const int rt = pick_pair_parts_rows(N1, K1, N2, K2, M, &p1, &p2);
    // (Workgroups of six waves are one a compute unit and fill the chip: attention's would take the places of the second product's, whose 71 blocks then
    // start late.  64 sequences of 60 keys, 71 heads on one, 4,544 x 4,544 and 4,544 x 18,176: 50 us, with workgroups of 128 rows 48.)
    return rt != PAIR_STATIONARY && rt != PAIR_SIX && (long)std::max(K1, K2) * 32 * 2 < LDS_PAST;
}

// What decides whether the products of such a launch hide the attention (`tuning.late_pays` has the lines): rounds, the workgroups a compute unit has
// at most, and slack, the blocks (64 elements of K by 64 rows of W, a third of a microsecond each, as a unit pulls some 25 GB/s) that a unit has more of the
// first product's than of the second's, which wait for attention.
extern "C" int pta_gemm_splitk_pair_attn_room(int N1, int K1, int N2, int K2, int M, int* rounds, int* slack) {
    if (N1 <= 0 || K1 <= 0 || N2 <= 0 || K2 <= 0 || M <= 0) return pta_fail("gemm_splitk_pair_attn_room: sizes must be positive");
    int p1, p2;
    const int rt = pick_pair_parts_rows(N1, K1, N2, K2, M, &p1, &p2);
    *rounds = *slack = 0;
    if (rt == PAIR_STATIONARY || rt == PAIR_SIX) return 0;
    const SplitkProblem a = make_problem(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, N1, K1, 0, 0, rt, p1, 0);
    const SplitkProblem b = make_problem(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, N2, K2, 0, 0, rt, p2, 0);
    const int units = max(1, pta_compute_units());
    *rounds = (a.tiles * a.parts + b.tiles * b.parts + units - 1) / units;
    *slack = *rounds * rt * (a.blocks_per_part - b.blocks_per_part);
    return 0;
}

// The pair with the attention that its second product takes (x2 [M, nh d] is written here): pta_attn_mfma of one token a sequence,
// whole contexts, `waves` (1 or 4) on a piece's keys; sync: groups of sixteen heads x nkv x M zeros; owners: -1, or how many of attention's
// workgroups the launch is to begin with (the products' do the others).
extern "C" int pta_gemm_splitk_pair_attn(float* part1, const void* x1, const void* W1, int N1, int K1, float* part2, void* x2,
                                         const void* W2, int N2, int K2, int M, const void* q, const void* k_pool, const void* v_pool,
                                         const int* block_table, int bt_stride, const int* cu_tokens, const int* seq_start,
                                         const PtaScoreBias* score_bias, int nh, int nkv, int d, float scale, const float* sink, int waves,
                                         int* sync, int owners, void* stream) {
    PTA_REQUIRE(waves == 1 || waves == RIDE_WAVES, "gemm_splitk_pair_attn: 1 or %d waves on the keys of a piece, got %d", RIDE_WAVES, waves);
    if (check_splitk("gemm_splitk_pair_attn", x1, W1, M, N1, K1)) return 1;
    if (check_splitk("gemm_splitk_pair_attn", x2, W2, M, N2, K2)) return 1;
    PTA_REQUIRE(pta_gemm_splitk_pair_attn_ok(N1, K1, N2, K2, M, nh, nkv, d), "gemm_splitk_pair_attn: no launch for %d rows by %d x %d and %d x %d, %d heads on %d of %d",
                M, N1, K1, N2, K2, nh, nkv, d);
    PTA_REQUIRE(part1 && part2 && sync && q && k_pool && v_pool && block_table && cu_tokens && seq_start, "gemm_splitk_pair_attn: null pointer");
    for (const void* p : {q, k_pool, v_pool, (const void*)x2})
        PTA_REQUIRE((uintptr_t)p % 16 == 0, "gemm_splitk_pair_attn: pointers must be 16-byte aligned");
    int bias_mode = 0;
    if (pta_score_bias_mode("gemm_splitk_pair_attn", score_bias, &bias_mode)) return 1;
    const float* slopes = score_bias ? score_bias->slopes : nullptr;
    int p1, p2;
    const int rt = pick_pair_parts_rows(N1, K1, N2, K2, M, &p1, &p2);
    const SplitkProblem a = make_problem(nullptr, part1, x1, W1, nullptr, nullptr, nullptr, N1, K1, 0, 0, rt, p1, 0);
    const SplitkProblem b = make_problem(nullptr, part2, x2, W2, nullptr, nullptr, nullptr, N2, K2, 0, 0, rt, p2, 0);
    AttnRide ride{};
    ride.attn = AttnArgs{(const bf16_t*)q, (const bf16_t*)k_pool, (const bf16_t*)v_pool, block_table, cu_tokens, seq_start, bt_stride, nh, nkv,
                         AttnMore{M, 1, 0, bias_mode, 0, 0, scale * PTA_LOG2E, slopes ? PTA_LOG2E * score_bias->scale : 0.f, slopes, (bf16_t*)x2,
                                  nullptr, nullptr, nullptr, sink, pta_head_rows_of(nullptr, nh, d)}};
    ride.groups = (nh / nkv + 15) / 16;
    ride.n_seqs = M;
    const int pieces = ride.groups * nkv * M;
    ride.tasks = waves == 1 ? (pieces + RIDE_WAVES - 1) / RIDE_WAVES : pieces;
    ride.owners = owners < 0 || owners > ride.tasks ? ride.tasks : owners;
    ride.sync = sync;
    return pta_splitk_attn_launch(a, b, M, rt, rotated(a, b), rotation_stride(), waves > 1, ride, (hipStream_t)stream);
}

// The same pair run to the end: y1 = act1(x1 . W1^T + bias1), y2 = act2(x2 . W2^T + bias2) in bfloat16; the two
// products share the matrix launch and the launch that adds their partial sums.
extern "C" int pta_gemm_splitk_pair_reduced_bf16(void* y1, float* part1, const void* x1, const void* W1,
                                                 const float* bias1, int N1, int K1, int act1, void* y2, float* part2,
                                                 const void* x2, const void* W2, const float* bias2, int N2, int K2,
                                                 int act2, int M, void* stream) {
    PTA_REQUIRE(y1 && y2, "gemm_splitk_pair_reduced_bf16: null output");
    PTA_REQUIRE(pta_act_known(act1) && pta_act_known(act2),
                "gemm_splitk_pair_reduced_bf16: unknown activation");
    const int rc = pta_gemm_splitk_pair_bf16(part1, x1, W1, N1, K1, part2, x2, W2, N2, K2, M, stream);
    if (rc) return rc;
    const long MN1 = (long)M * N1, MN2 = (long)M * N2;
    int P1, P2;
    pick_pair_parts_rows(N1, K1, N2, K2, M, &P1, &P2);
    hipLaunchKernelGGL(gemm_splitk_reduce2_kernel, dim3((unsigned)((MN1 + MN2 + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, (bf16_t*)y1, part1, bias1, MN1, N1, P1, act1, (bf16_t*)y2, part2, bias2, MN2, N2,
                       P2, act2);
    return pta_check_launch("gemm_splitk_pair_reduced_bf16");
}

// what the launches that take fused query_key_value rows to their end ask of their arguments
static int check_qkv_tail(const char* what, const void* q_out, const PtaRotation& rot,
                          const int* token_pos, const int* token_seq,
                          const int* block_table, const void* k_pool, const void* v_pool, int nh, int nkv, int d,
                          int layout, int write_cache) {
    PTA_REQUIRE(nh > 0 && nkv > 0 && d > 0 && nh % nkv == 0, "%s: heads %d, kv heads %d, head size %d", what, nh, nkv, d);
    if (pta_check_rotation(what, rot, d, token_seq)) return 1;
    PTA_REQUIRE(d % 2 == 0, "%s: head size %d must be even", what, d);
    PTA_REQUIRE(layout >= 0 && layout <= 2, "%s: unknown layout %d", what, layout);
    PTA_REQUIRE(layout != PTA_QKV_TAIL || nkv == 1, "%s: the tail layout has one kv head, got %d", what, nkv);
    PTA_REQUIRE(layout != PTA_QKV_INTERLEAVED || nkv == nh, "%s: the interleaved layout needs kv heads == heads", what);
    PTA_REQUIRE(q_out && token_pos, "%s: null pointer", what);
    PTA_REQUIRE(!write_cache || (k_pool && v_pool && block_table && token_seq), "%s: null cache pointer", what);
    return 0;
}

// The same pair with the first product a fused query_key_value projection taken to its end: queries rotated in
// q_out [M, heads, d], keys and values in the cache pages (as pta_qkv_rope_cache leaves them); even head sizes.
extern "C" int pta_gemm_splitk_pair_reduced_qkv_bf16(void* q_out, float* part1, const void* x1, const void* W1,
                                                     const float* bias1, int K1, const PtaRotation* rotation,
                                                     const int* token_pos, const int* token_seq, const int* block_table,
                                                     int bt_stride, void* k_pool, void* v_pool, int nh, int nkv, int d,
                                                     int layout, int write_cache, void* y2, float* part2, const void* x2,
                                                     const void* W2, const float* bias2, int N2, int K2, int act2, int M,
                                                     void* stream) {
    const PtaRotation rot = pta_rotation_of(rotation);
    if (check_qkv_tail("gemm_splitk_pair_reduced_qkv_bf16", q_out, rot, token_pos, token_seq, block_table, k_pool, v_pool, nh,
                       nkv, d, layout, write_cache))
        return 1;
    PTA_REQUIRE(y2, "gemm_splitk_pair_reduced_qkv_bf16: null pointer");
    PTA_REQUIRE(pta_act_known(act2), "gemm_splitk_pair_reduced_qkv_bf16: unknown activation %d", act2);
    const int N1 = (nh + 2 * nkv) * d;
    const int rc = pta_gemm_splitk_pair_bf16(part1, x1, W1, N1, K1, part2, x2, W2, N2, K2, M, stream);
    if (rc) return rc;
    const long MN1 = (long)M * N1, MN2 = (long)M * N2;
    int P1, P2;
    pick_pair_parts_rows(N1, K1, N2, K2, M, &P1, &P2);
    const QkvTail tail{(bf16_t*)q_out, rot, token_pos, token_seq, block_table, bt_stride, (bf16_t*)k_pool,
                       (bf16_t*)v_pool, nh, nkv, d, layout, write_cache};
    const bool four = N2 % 4 == 0 && (uintptr_t)part2 % 16 == 0 && (uintptr_t)y2 % 8 == 0;
    hipLaunchKernelGGL((four ? gemm_splitk_reduce2_qkv_kernel<4> : gemm_splitk_reduce2_qkv_kernel<1>),
                       dim3((unsigned)((MN1 / 2 + (four ? MN2 / 4 : MN2) + 255) / 256)), dim3(256), 0, (hipStream_t)stream, tail, part1, bias1, MN1, N1, P1, (bf16_t*)y2, part2, bias2, MN2, N2, P2, act2);
    return pta_check_launch("gemm_splitk_pair_reduced_qkv_bf16");
}

// A fused query_key_value projection on its own (17 to 256 rows), taken to its end by the launch that adds its
// partial sums: part [pta_gemm_splitk_parts(N, K, 0, 0), M, N] is the workspace, N = (nh + 2 nkv) d.
extern "C" int pta_gemm_splitk_reduced_qkv_bf16(void* q_out, float* part, const void* x, const void* W,
                                                const float* bias, int K, const PtaRotation* rotation,
                                                const int* token_pos, const int* token_seq, const int* block_table,
                                                int bt_stride, void* k_pool, void* v_pool, int nh, int nkv, int d,
                                                int layout, int write_cache, int M, void* stream) {
    const PtaRotation rot = pta_rotation_of(rotation);
    if (check_qkv_tail("gemm_splitk_reduced_qkv_bf16", q_out, rot, token_pos, token_seq, block_table, k_pool, v_pool, nh, nkv,
                       d, layout, write_cache))
        return 1;
    PTA_REQUIRE(part, "gemm_splitk_reduced_qkv_bf16: null workspace");
    const int N = (nh + 2 * nkv) * d;
    const int rc = pta_gemm_splitk_bf16(nullptr, part, x, W, nullptr, nullptr, nullptr, M, N, K, PTA_ACT_NONE, 0, 0, 0, 0,
                                        0, 0, stream);
    if (rc) return rc;
    const long MN = (long)M * N;
    const QkvTail tail{(bf16_t*)q_out, rot, token_pos, token_seq, block_table, bt_stride, (bf16_t*)k_pool,
                       (bf16_t*)v_pool, nh, nkv, d, layout, write_cache};
    hipLaunchKernelGGL(gemm_splitk_reduce2_qkv_kernel<1>, dim3((unsigned)((MN / 2 + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, tail, part, bias, MN, N, pta_gemm_splitk_parts(N, K, 0, 0), (bf16_t*)nullptr,
                       (const float*)nullptr, (const float*)nullptr, 0L, 1, 1, 0);
    return pta_check_launch("gemm_splitk_reduced_qkv_bf16");
}

// ---- the same product for callers that cannot allocate ---------------------------------------------------
// The 32-bit partial sums of the ranges of K lie in a file-scope device array instead of a workspace that the
// caller brings.  Every GPU holds its own copy of the array at its own address until the process ends; its
// address is asked from the runtime once per device, with that device current, and only that address is ever
// handed to a kernel or a runtime call (the array's name in host code is a stand-in, no device address).
#define PTA_STATIC_PART_FLOATS (4 * 1024 * 1024)  // 16 MiB per GPU
#define PTA_MAX_DEVICES 64
static __device__ __align__(256) float scratch[PTA_STATIC_PART_FLOATS];
static float* scratch_ptr[PTA_MAX_DEVICES] = {nullptr};
static std::mutex scratch_lock;

// the current device's copy of `scratch`; null after storing the reason
static float* static_workspace() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= PTA_MAX_DEVICES) {
        pta_fail("gemm_splitk_bf16_static: no current device (or more than %d devices)", PTA_MAX_DEVICES);
        return nullptr;
    }
    std::lock_guard<std::mutex> hold(scratch_lock);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            pta_fail("gemm_splitk_bf16_static: the workspace's address on device %d is not known: %s", dev,
                     hipGetErrorString(e));
            return nullptr;
        }
        scratch_ptr[dev] = (float*)p;
    }
    return scratch_ptr[dev];
}

extern "C" long pta_gemm_splitk_static_floats(void) { return PTA_STATIC_PART_FLOATS; }

extern "C" int pta_gemm_splitk_bf16_static(void* y, const void* x, const void* W, const float* bias, const void* add1,
                                           const void* add2, int M, int N, int K, int act, int out_f32, void* stream) {
    if (check_splitk("gemm_splitk_bf16_static", x, W, M, N, K)) return 1;
    const long need = (long)pta_gemm_splitk_parts(N, K, 0, 0) * M * N;
    PTA_REQUIRE(need <= (long)PTA_STATIC_PART_FLOATS,
                "gemm_splitk_bf16_static: %d ranges of K x %d rows x %d features are %ld partial sums, the built-in "
                "workspace holds %d (bring a workspace to pta_gemm_splitk_bf16 instead)",
                pta_gemm_splitk_parts(N, K, 0, 0), M, N, need, PTA_STATIC_PART_FLOATS);
    float* part = static_workspace();
    if (!part) return 1;
    // every partial sum that the reduction reads is written by this call's matrix launch first, so nothing of
    // the array has to start at zero
    return pta_gemm_splitk_bf16(y, part, x, W, bias, add1, add2, M, N, K, act, out_f32, 0, 0, 0, 0, 1, stream);
}
