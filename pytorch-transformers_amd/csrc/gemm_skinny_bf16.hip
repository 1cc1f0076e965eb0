// y[M,N] = act(x[M,K] . W[N,K]^T + bias) + add1 + add2 for few rows (M <= 64), bfloat16 in,
// 32-bit accumulation on the matrix cores.  This is the decode step's linear layer: the work is
// reading W once from HBM, so the kernel is laid out for that, not for the arithmetic.
//
// A workgroup of S waves owns 16*RT rows of W and all of K.  Its waves take the 64-element K-steps
// round robin (wave w: steps w, w + S, ...), so neighbouring waves read neighbouring 128-byte lines
// of the same rows.  Up to sixteen rows of x (64 with a small matrix) a wave brings whole lines of its rows of W and of x straight to a
// ring of its own in LDS, several steps ahead, and reads the operands of v_mfma_f32_16x16x32_bf16 from there (lds_stream.h: why, and what
// it measured).  More rows of x, and rows of W too long for the buffers' offsets, go by registers: a wave works in
// stages of U steps and always has the next stage's loads in flight while the matrix cores consume the current one (two
// register buffers); W rows are the A operand (lane: row = lane % 16, eight consecutive k at (lane / 16) * 8, one
// 16-byte load straight from global memory), x rows are the B operand (same shape, buffer loads whose
// bounds are the M real rows, so the padding rows of the tile read zeros and cost no traffic).  The S partial tiles are summed through
// LDS in wave order, then bias, activation and additions are applied and the tile is stored.  S is chosen from N and K alone, so
// the order of summation never depends on M or on what else is in the batch.
//
// What is left between a launch and the rate of its loads (22,848 x 4,544, one row, 207 MB: 38.2 us from launch to launch): workgroups start
// within 0.5 us and set up for 0.5, their rings end between 26 and 36 us after the first start (5.9 TB/s over the whole), sums and store take 0.8,
// and the next launch starts 1.1 later.  One load of x a step instead of two, where x has eight rows or fewer, changed nothing.
#include "common.h"
#include "glu.h"
#include "lds_stream.h"
#include "pta_kernels.h"
#include "qkv_tail.h"

#include <stdlib.h>

#include <algorithm>
#include <type_traits>

union Frag {
    uint4 u;
    bf16x8_t v;
    i32x4_t i;
};

template <typename OutT> struct OutIo;
template <> struct OutIo<float> {
    static __device__ __forceinline__ float round(float v) { return v; }
    static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
};
template <> struct OutIo<bf16_t> {
    static __device__ __forceinline__ float round(float v) { return round_to_bf16(v); }
    static __device__ __forceinline__ void st(bf16_t* p, float v) { *p = f32_to_bf16_bits(v); }
};

template <int MT, int RT, int U>
struct Stage {
    Frag a[U][2][RT];
    Frag b[U][2][MT];
    uint32_t keep[U][2];  // all ones if the chunk lies inside K, else zero
};

// Loads are unconditional: the address is clamped into the row, and the data of a chunk past K is
// masked to zero only when it is used.  A load under a branch, or a mask applied here, would make
// the wave wait for loads it has just issued, and the two stages would no longer overlap.
template <int MT, int RT, int U>
__device__ __forceinline__ void load_stage(Stage<MT, RT, U>& st, const bf16_t* const (&wrow)[RT],
                                           __amdgpu_buffer_rsrc_t xres, int r, int first_step, int S, int g, int K,
                                           int nsteps, int rot) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        // the workgroup walks K from its own starting step and wraps round; steps past the last are masked
        int step = first_step + u * S;
        if (step < nsteps) { step += rot; step -= step >= nsteps ? nsteps : 0; }
        const int k0 = step * 64 + g * 8;  // K % 8 == 0: a chunk of 8 is inside K or outside it
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const int k = k0 + hf * 32;
            const int kc = min(k, K - 8);
            st.keep[u][hf] = k < K ? 0xffffffffu : 0u;
#pragma unroll
            for (int t = 0; t < RT; ++t) st.a[u][hf][t].u = *reinterpret_cast<const uint4*>(wrow[t] + kc);
#pragma unroll
            for (int t = 0; t < MT; ++t)  // a row past M lies outside the buffer's bounds: it reads zeros and costs no traffic
                st.b[u][hf][t].i = __builtin_amdgcn_raw_buffer_load_b128(xres, ((t * 16 + r) * K + kc) * 2, 0, 0);
        }
    }
}

template <int MT, int RT, int U>
__device__ __forceinline__ void compute_stage(const Stage<MT, RT, U>& st, f32x4_t (&acc)[RT][MT]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                Frag a = st.a[u][hf][rt];
                const uint32_t keep = st.keep[u][hf];
                a.u.x &= keep; a.u.y &= keep; a.u.z &= keep; a.u.w &= keep;
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, st.b[u][hf][mt].v, acc[rt][mt], 0, 0, 0);
            }
}

// A wave's steps of K, two stages of registers in turn: rows of W from the lane's addresses, so rows of any length
template <int MT, int RT, int U>
__device__ __forceinline__ void by_registers(f32x4_t (&acc)[RT][MT], const bf16_t* const (&wrow)[RT], const bf16_t* x, int lane, int wave,
                                             int S, int M, int K, int nsteps, int rot) {
    // x through a buffer descriptor whose bounds are the M real rows (0x00020000: 32-bit raw data format)
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, M * K * 2, 0x00020000);
    const int r = lane & 15, g = lane >> 4;
    Stage<MT, RT, U> s0, s1;
    load_stage<MT, RT, U>(s0, wrow, xres, r, wave, S, g, K, nsteps, rot);
    // the scheduling barriers keep the compiler from sinking a stage's loads down to their first
    // use, which would shrink what is in flight to a load or two
    for (int step = wave; step < nsteps; step += 2 * U * S) {
        load_stage<MT, RT, U>(s1, wrow, xres, r, step + U * S, S, g, K, nsteps, rot);
        __builtin_amdgcn_sched_barrier(0);
        compute_stage<MT, RT, U>(s0, acc);
        __builtin_amdgcn_sched_barrier(0);
        load_stage<MT, RT, U>(s0, wrow, xres, r, step + 2 * U * S, S, g, K, nsteps, rot);
        __builtin_amdgcn_sched_barrier(0);
        compute_stage<MT, RT, U>(s1, acc);
        __builtin_amdgcn_sched_barrier(0);
    }
}

#define SHARE_BITS 26
#define SHARE_MOST 63  // in the bits above

// How `items` (rows of W, pairs of them) are shared out evenly to `groups` workgroups: the first `over` have one more than the others.
// Made on the host: the division by a number of workgroups was 300 instructions at the start of a launch of few microseconds.
// In a launch's arguments it is a word, `each` in the six highest bits and `over` in the others: a group has up to 64 items, so 64 for every one is said as 63
// and one more for all of them, and a launch has fewer groups than 2^26 (of a wave each: 2^32 threads).
struct Share {
    int each, over;
    Share() = default;
    Share(int items, int groups) : each(groups > 0 ? items / groups : 0), over(groups > 0 ? items % groups : 0) {
        if (each == SHARE_MOST + 1 && over == 0) each = SHARE_MOST, over = groups;
    }
    __host__ __device__ __forceinline__ int begin(int j) const { return j * each + (j < over ? j : over); }
    __host__ __device__ __forceinline__ int end(int j) const { return begin(j) + each + (j < over ? 1 : 0); }
    bool fits() const { return each <= SHARE_MOST && over < 1 << SHARE_BITS; }
    uint32_t packed() const { return (uint32_t)each << SHARE_BITS | (uint32_t)over; }
    static __host__ __device__ __forceinline__ Share of(uint32_t word) {
        Share s;
        s.each = word >> SHARE_BITS, s.over = word & ((1u << SHARE_BITS) - 1);
        return s;
    }
};

// Where workgroup j of `groups` finds its share of `items` to begin and end, as a launch's word says it.
extern "C" int pta_gemm_skinny_share(int items, int groups, int j, int* begin, int* end) {
    PTA_REQUIRE(items > 0 && groups > 0 && j >= 0 && j < groups, "gemm_skinny_share: workgroup %d of %d for %d items", j, groups, items);
    const Share made(items, groups);
    PTA_REQUIRE(made.fits(), "gemm_skinny_share: %d items for each of %d workgroups are more than a word says", items / groups, groups);
    const Share read = Share::of(made.packed());
    *begin = read.begin(j), *end = read.end(j);
    return 0;
}

// The kernels here take what their loads of W and x are found by first, in the fourteen words that are in registers when a workgroup starts: the
// arguments behind them are a load away, 0.7 us over cold caches, and what is asked for at the front the first loads wait for.  (With the problem's struct
// first, 24 layers of four such launches, 1,040 wide, 24 steps of 5 rows: 21.8 ms, this way 21.0: 0.35 us a launch.)  How a workgroup walks, in a word: its waves, a head's elements (with a QkvTail; the sign: its pairs are
// those that lie half a head apart), and where in K it starts.
struct Walk {
    int waves, d, rot_stride;
    bool plain;
    static uint32_t packed(int waves, int rot_stride, int d = 0, bool plain = false) {
        return (uint32_t)waves | (uint32_t)d << 4 | (plain ? 1u << 15 : 0u) | (uint32_t)rot_stride << 16;
    }
    __device__ __forceinline__ Walk(uint32_t word)
        : waves(word & 15), d(word >> 4 & 0x7ff), rot_stride(word >> 16), plain((word >> 15 & 1) != 0) {}
};

// where a workgroup starts in K, for rows of W a power of two long (gemm_skinny_kernel)
__device__ __forceinline__ int start_step(int rot_stride, int nsteps) {
    return rot_stride > 0 ? (int)((unsigned)(blockIdx.x * rot_stride) % (unsigned)nsteps) : 0;
}

// One product of a launch: a launch may carry two that share M and K (a block's two input projections),
// so that the second one's workgroups fill the chip while the first one's drain.
struct SkinnyProblem {
    void* y;
    const bf16_t* x;
    const bf16_t* W;
    const float* bias;
    const bf16_t* add1;
    const bf16_t* add2;
    int N;
    int act;
    int blocks;  // workgroups of this product
    Share rows;  // of W, over them (pairs of rows where a launch works on those)
};

// what follows the product, for one feature: bias, activation, additions
template <typename OutT>
__device__ __forceinline__ void store_feature(OutT* y, const float* bias, int act, const bf16_t* add1, const bf16_t* add2, int N, int m,
                                              int n, float sum) {
    float v = OutIo<OutT>::round(sum);
    if (bias) v = OutIo<OutT>::round(v + bias[n]);
    // (the others run as a pass of their own, as squared ReLU did: 4.7 us behind a product of 10, 8,192 x 2,048)
    if (act == PTA_ACT_GELU) v = sizeof(OutT) == 2 ? gelu_bf16(v) : gelu_erf(v);
    else if (act == PTA_ACT_RELU2) v = apply_act_bf16(v, PTA_ACT_RELU2);
    const long o = (long)m * N + n;
    if (add1) v += bf16_bits_to_f32(add1[o]);
    if (add2) v += bf16_bits_to_f32(add2[o]);
    OutIo<OutT>::st(y + o, v);
}

// With a QkvTail (qkv_tail.h) the first product's rows are not stored: they are split into heads, rotated and written
// as queries and into the cache pages.  The rotation works on pairs of a head's elements, so a workgroup takes the
// first elements of sixteen pairs as its first row tile and their partners as its second (TAIL 1: whole heads in
// half-split pairs, or no rotation: pair p is elements p and p + d/2, and four pairs in a row are stored as eight
// bytes; TAIL 2: any rotation that qkv_tail_pair_elements describes, stored element by element).
template <int MT, int RT, int U, typename OutT, int TAIL = 0, int D = 0>
__global__ __launch_bounds__(512) void gemm_skinny_kernel(const bf16_t* __restrict__ xa, const bf16_t* __restrict__ Wa, const bf16_t* __restrict__ xb,
                                                          const bf16_t* __restrict__ Wb, int M, int K, int blocks_a, uint32_t share_a,
                                                          uint32_t share_b, uint32_t how, SkinnyProblem pa, SkinnyProblem pb, QkvTail tail) {
    static_assert(!TAIL || (RT == 2 && MT == 1 && sizeof(OutT) == 2), "the query_key_value tail: two row tiles, sixteen rows of x");
    static_assert(D == 0 || MT == 1, "through LDS: sixteen rows of x");
    // the waves' sums, [RT][MT][64] each; through LDS they take the place of the waves' rings
    extern __shared__ __attribute__((aligned(1024))) f32x4_t part[];
    constexpr int WAVE = D == 0 ? RT * MT * 64 : RowStream<RT, D == 0 ? 1 : D>::RING / 16;
    const Walk walk(how);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, S = walk.waves, head = walk.d;
    const int r = lane & 15;
    const bool second = (int)blockIdx.x >= blocks_a;
    const bf16_t* __restrict__ x = second ? xb : xa;
    const bf16_t* __restrict__ W = second ? Wb : Wa;
    // the workgroups of a product share its rows evenly: this one has rows n0 .. n1 - 1, at most 16 * RT
    const int j = (int)blockIdx.x - (second ? blocks_a : 0);
    const Share mine = Share::of(second ? share_b : share_a);
    const int n0 = mine.begin(j), n1 = mine.end(j);
    const bool tailed = TAIL && !second;
    // with the tail: workgroup j has pairs s16*16 .. +15 of segment seg (a head's q, k or v); their elements are its two row tiles
    const int per_seg = TAIL ? head / 32 : 1, seg = j / per_seg, s16 = j % per_seg;
    auto tail_row = [&](int i, int t) {  // element t of pair i of the sixteen, within the segment
        if (TAIL == 1) return s16 * 16 + i + (t & 1) * (head >> 1);
        int e[2] = {0, 0};
        bool rotated;
        qkv_tail_pair_elements(tail.rot, tail.d, s16 * 16 + i, e[0], e[1], rotated);
        return t & 1 ? e[1] : e[0];
    };
    f32x4_t acc[RT][MT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int nsteps = (K + 63) >> 6;
    // Where a row of W is a power of two long, every workgroup walking K from its start would ask the same few
    // memory channels at the same time (K = 4,096: 13 % slower than K = 4,160).  So each starts `rot_stride`
    // steps after its neighbour.  A feature's order of summation follows from N, K and the launch alone.
    const int rot = start_step(walk.rot_stride, nsteps);
    if constexpr (D > 0) {
        RowStream<RT, D> rows;
        rows.x = buffer_of(x, M * K * 2);
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int first = tailed ? seg * head : min(n0 + t * 16, n1 - 1), count = tailed ? head : min(16, n1 - n0 - t * 16);
            rows.w[t] = buffer_of(W + (long)first * K, max(count, 0) * K * 2);
#pragma unroll
            for (int l = 0; l < 2; ++l) {
                const int i = stream_row(lane, l), row = tailed ? tail_row(i, t) : i;
                rows.w_at[2 * t + l] = row < count ? row * K * 2 : LDS_PAST;
            }
        }
#pragma unroll
        for (int l = 0; l < 2; ++l) rows.x_at[l] = stream_row(lane, l) < M ? stream_row(lane, l) * K * 2 : LDS_PAST;
        f32x4_t sums[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) sums[rt] = acc[rt][0];
        rows.run(sums, (const char*)(part + wave * WAVE), lane, wave, S, K, nsteps, rot);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt][0] = sums[rt];
    } else {
        const bf16_t* wrow[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) wrow[t] = W + (long)(tailed ? seg * head + tail_row(r, t) : min(n0 + t * 16 + r, n1 - 1)) * K;
        by_registers<MT, RT, U>(acc, wrow, x, lane, wave, S, M, K, nsteps, rot);
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) part[wave * WAVE + (rt * MT + mt) * 64 + lane] = acc[rt][mt];
    __syncthreads();

    OutT* __restrict__ y = (OutT*)(second ? pb.y : pa.y);
    const float* __restrict__ bias = second ? pb.bias : pa.bias;
    const bf16_t* __restrict__ add1 = second ? pb.add1 : pa.add1;
    const bf16_t* __restrict__ add2 = second ? pb.add2 : pa.add2;
    const int N = second ? pb.N : pa.N, act = second ? pb.act : pa.act;
    if constexpr (TAIL) {
        if (tailed) {
            // thread ln: token m = ln % 16, features i0 .. i0+3 of the segment's lower half and their partners
            for (int ln = threadIdx.x; ln < 64; ln += S * 64) {
                f32x4_t lo = part[ln], hi = part[64 + ln];
                for (int w = 1; w < S; ++w) {
                    const f32x4_t p = part[w * WAVE + ln], q = part[w * WAVE + 64 + ln];
                    lo[0] += p[0]; lo[1] += p[1]; lo[2] += p[2]; lo[3] += p[3];
                    hi[0] += q[0]; hi[1] += q[1]; hi[2] += q[2]; hi[3] += q[3];
                }
                const int m = ln & 15;
                if (m >= M) continue;
                const int d = tail.d, half = d >> 1, i0 = s16 * 16 + (ln >> 4) * 4;
                if constexpr (TAIL == 2) {  // pairs i0 .. i0+3, wherever their elements lie
#pragma unroll
                    for (int e = 0; e < 4; ++e) qkv_tail_pair(tail, bias, m, seg, i0 + e, round_to_bf16(lo[e]), round_to_bf16(hi[e]));
                    continue;
                }
                int kind, head;  // 0 query, 1 key, 2 value
                qkv_tail_segment(tail, seg, kind, head);
                if (kind != 0 && !tail.write_cache) continue;
                const int pos = tail.token_pos[m];
                float a[4], b[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    a[e] = round_to_bf16(lo[e]);
                    b[e] = round_to_bf16(hi[e]);
                    if (bias) {
                        a[e] = round_to_bf16(a[e] + bias[seg * d + i0 + e]);
                        b[e] = round_to_bf16(b[e] + bias[seg * d + half + i0 + e]);
                    }
                }
                if (tail.rot.inv_freq && kind != 2) {
                    const float* freq = qkv_tail_freq(tail, m);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float ang = (float)pos * freq[i0 + e];
                        const float c = cosf(ang) * tail.rot.cs_scale, sn = sinf(ang) * tail.rot.cs_scale;
                        const float x0 = a[e], x1 = b[e];
                        a[e] = x0 * c - x1 * sn;
                        b[e] = x1 * c + x0 * sn;
                    }
                }
                uint2 pa4, pb4;
                pa4.x = (uint32_t)f32_to_bf16_bits(a[0]) | ((uint32_t)f32_to_bf16_bits(a[1]) << 16);
                pa4.y = (uint32_t)f32_to_bf16_bits(a[2]) | ((uint32_t)f32_to_bf16_bits(a[3]) << 16);
                pb4.x = (uint32_t)f32_to_bf16_bits(b[0]) | ((uint32_t)f32_to_bf16_bits(b[1]) << 16);
                pb4.y = (uint32_t)f32_to_bf16_bits(b[2]) | ((uint32_t)f32_to_bf16_bits(b[3]) << 16);
                if (kind == 0) {
                    bf16_t* dst = tail.q_out + ((long)m * tail.nh + head) * d + i0;
                    *reinterpret_cast<uint2*>(dst) = pa4;
                    *reinterpret_cast<uint2*>(dst + half) = pb4;
                    continue;
                }
                const long page = tail.block_table[(long)tail.token_seq[m] * tail.bt_stride + pos / PTA_PAGE];
                const int in_page = pos % PTA_PAGE;
                if (kind == 1) {
                    bf16_t* dst = tail.k_pool + ((page * tail.nkv + head) * PTA_PAGE + in_page) * (long)d + i0;
                    *reinterpret_cast<uint2*>(dst) = pa4;
                    *reinterpret_cast<uint2*>(dst + half) = pb4;
                } else {
                    bf16_t* dst = tail.v_pool + ((page * tail.nkv + head) * (long)d + i0) * PTA_PAGE + in_page;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        dst[(long)e * PTA_PAGE] = f32_to_bf16_bits(a[e]);
                        dst[(long)(half + e) * PTA_PAGE] = f32_to_bf16_bits(b[e]);
                    }
                }
            }
            return;
        }
    }
    // item (rt, mt, ln): outputs of row m = mt*16 + ln%16, columns n0 + rt*16 + (ln/16)*4 + 0..3
    for (int item = threadIdx.x; item < RT * MT * 64; item += S * 64) {
        const int ln = item & 63, mt = (item >> 6) % MT, rt = (item >> 6) / MT;
        f32x4_t sum = part[(rt * MT + mt) * 64 + ln];
        for (int w = 1; w < S; ++w) {
            const f32x4_t p = part[w * WAVE + (rt * MT + mt) * 64 + ln];
            sum[0] += p[0]; sum[1] += p[1]; sum[2] += p[2]; sum[3] += p[3];
        }
        const int m = mt * 16 + (ln & 15);
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + rt * 16 + (ln >> 4) * 4 + i;
            if (n < n1) store_feature<OutT>(y, bias, act, add1, add2, N, m, n, sum[i]);
        }
    }
}

// the two elements of a rotation pair, within their head
__device__ __forceinline__ void tail_elements(const Walk& walk, const QkvTail& tail, int pair, int (&e)[2]) {
    bool rotated;
    if (walk.plain) {
        e[0] = pair, e[1] = pair + (walk.d >> 1);
        return;
    }
    asm volatile("");  // (a branch: what is read there is not among the first arguments)
    qkv_tail_pair_elements(tail.rot, walk.d, pair, e[0], e[1], rotated);
}

// Heads that hold rotation pairs p0 .. p1 - 1, `half` pairs a head: what a workgroup's buffer of W has to span.  Two for up to eight
// pairs of heads of fourteen elements and more; eight pairs of heads of two lie in eight.
__device__ __forceinline__ int heads_of(int p0, int p1, int half) { return (p1 - 1) / half - p0 / half + 1; }

// A fused query_key_value product on its own, taken to its end by its epilogue (qkv_tail.h), for matrices whose rows are spread
// over all compute units (``launch_skinny``): a workgroup has up to eight neighbouring rotation pairs, the first elements as
// rows 0 .. 7 of its one tile, their partners as rows 8 .. 15.  Bound by the launch, not by W: at 3,120 x 1,040 and 5 rows it
// takes what the product alone takes, and the launch that split, rotated and wrote the cache (4 us a layer) is gone: a
// model of 24 such layers, 5 sequences, 24 steps and their prompts 34.5 -> 32.2 ms.
template <int D>
__global__ __launch_bounds__(512) void gemm_skinny_tail_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, int M, int K,
                                                               uint32_t items, uint32_t how, const float* __restrict__ bias, QkvTail tail) {
    extern __shared__ __attribute__((aligned(1024))) f32x4_t part[];  // the waves' rings, and then their sums
    constexpr int WAVE = D == 0 ? 64 : RowStream<1, D == 0 ? 1 : D>::RING / 16;
    const Walk walk(how);
    const Share share = Share::of(items);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, S = walk.waves, head = walk.d, half = head >> 1;
    const int p0 = share.begin(blockIdx.x), p1 = share.end(blockIdx.x);
    const int nsteps = (K + 63) >> 6, rot = start_step(walk.rot_stride, nsteps);
    auto row_of = [&](int pair, int second) {  // of W: an element of a pair
        int e[2];
        tail_elements(walk, tail, pair % half, e);
        return pair / half * head + (second ? e[1] : e[0]);
    };
    f32x4_t sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if constexpr (D > 0) {
        const int first = p0 / half * head;  // row of W that the others are counted from
        RowStream<1, D> rows;
        rows.w[0] = buffer_of(W + (long)first * K, heads_of(p0, p1, half) * head * K * 2);
        rows.x = buffer_of(x, M * K * 2);
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            const int pair = p0 + (lane >> 3);
            rows.w_at[l] = pair < p1 ? (row_of(pair, l) - first) * K * 2 : LDS_PAST;
            rows.x_at[l] = stream_row(lane, l) < M ? stream_row(lane, l) * K * 2 : LDS_PAST;
        }
        f32x4_t acc[1] = {sum};
        rows.run(acc, (const char*)(part + wave * WAVE), lane, wave, S, K, nsteps, rot);
        sum = acc[0];
    } else {  // (places past the end read a pair again)
        const bf16_t* wrow[1] = {W + (long)row_of(min(p0 + (lane & 7), p1 - 1), lane >> 3 & 1) * K};
        f32x4_t acc[1][1] = {{sum}};
        by_registers<1, 1, 2>(acc, wrow, x, lane, wave, S, M, K, nsteps, rot);
        sum = acc[0][0];
    }
    part[wave * WAVE + lane] = sum;
    __syncthreads();
    const float* sums = (const float*)part;  // row i of the tile, column m: lane (i / 4) * 16 + m, element i % 4
    for (int item = threadIdx.x; item < 128; item += S * 64) {
        const int m = item & 15, i = item >> 4, pair = p0 + i;
        if (m >= M || pair >= p1) continue;
        const int at = ((i >> 2) * 16 + m) * 4 + (i & 3);
        float a = sums[at], b = sums[at + 2 * 16 * 4];
        for (int w = 1; w < S; ++w) a += sums[w * WAVE * 4 + at], b += sums[w * WAVE * 4 + at + 2 * 16 * 4];
        qkv_tail_pair(tail, bias, m, pair / half, pair % half, round_to_bf16(a), round_to_bf16(b));
    }
}

// What follows the halves kernels' sums: `sums` of wave w from w * stride on, items n0 .. n1 - 1 (rows, or rotation pairs)
template <bool DIAG, typename OutT, bool TAIL>
__device__ __forceinline__ void halves_end(const SkinnyProblem& p, const QkvTail& tail, const float* sums, int stride, int S, int M, int n0, int n1) {
    const int half = TAIL ? tail.d >> 1 : 1;
    auto sum_of = [&](int m, int i) {  // row i of the eight for row m of x
        constexpr int OTHER = (32 + (DIAG ? 8 : 0)) * 4;
        const int at = ((m >> 4) * 64 + (i >> 2) * 16 + (m & 15)) * 4 + (i & 3);
        float v = sums[at] + sums[at + OTHER];
        for (int w = 1; w < S; ++w) {
            v += sums[w * stride + at];
            v += sums[w * stride + at + OTHER];
        }
        return v;
    };
    if constexpr (TAIL) {
        for (int item = threadIdx.x; item < 4 * M; item += S * 64) {
            const int m = item >> 2, i = item & 3, pair = n0 + i;
            if (pair < n1) qkv_tail_pair(tail, p.bias, m, pair / half, pair % half, round_to_bf16(sum_of(m, i)), round_to_bf16(sum_of(m, i + 4)));
        }
    } else {
        for (int item = threadIdx.x; item < 8 * M; item += S * 64) {
            const int m = item >> 3, i = item & 7;
            if (n0 + i < n1) store_feature<OutT>((OutT*)p.y, p.bias, p.act, p.add1, p.add2, p.N, m, n0 + i, sum_of(m, i));
        }
    }
}

// Small matrices, eight rows of W or fewer a workgroup (N up to eight times the compute units): what bounds such a launch, apart
// from its start, is not memory but the compute units' address paths, a wave's load taking sixteen cycles whatever it fetches,
// and with eight rows in a tile of sixteen half of W's loads fetched nothing new.  So a tile is eight rows at two places of K:
// lanes of rows 0 .. 7 carry 64 elements of a step of 128, lanes of rows 8 .. 15 the 64 behind them.  With up to eight rows
// of x (DIAG) x is laid out the same way, and one matrix instruction makes both halves' sums, in the blocks on its
// diagonal; with more, two instructions do, and of each the half that belongs together is kept.  Either way a sum is that of
// the first halves of its wave's steps plus that of the second, the waves' in order: the same bits for any number of rows.
// TAIL: a fused query_key_value product taken to its end as by gemm_skinny_tail_kernel; rows 0 .. 3 are the first elements of up
// to four rotation pairs, rows 4 .. 7 their partners.
template <int MT, bool DIAG, int U, typename OutT, bool TAIL>
__global__ __launch_bounds__(512) void gemm_skinny_halves_kernel(const bf16_t* __restrict__ x_rows, const bf16_t* __restrict__ W, int M, int K, uint32_t items,
                                                                 uint32_t how, SkinnyProblem p, QkvTail tail) {
    static_assert(!DIAG || MT == 1, "both halves of K in a tile: eight rows of x");
    constexpr int BT = DIAG ? 1 : 2 * MT;  // fragments of x a half step
    extern __shared__ f32x4_t part[];      // [S][MT][64]
    const Walk walk(how);
    const Share share = Share::of(items);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, S = walk.waves;
    const int r = lane & 15, g = lane >> 4, row = r & 7, sub = r >> 3;
    const int half = TAIL ? walk.d >> 1 : 1;
    const int n0 = share.begin(blockIdx.x), n1 = share.end(blockIdx.x);  // pairs, or rows
    int w_row = min(n0 + row, n1 - 1);
    if (TAIL) {
        const int mine = min(n0 + (row & 3), n1 - 1);  // (places past the end read a pair again)
        int e[2];
        tail_elements(walk, tail, mine % half, e);
        w_row = mine / half * walk.d + (row < 4 ? e[0] : e[1]);
    }
    const bf16_t* wrow = W + (long)w_row * K;
    __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)x_rows, 0, M * K * 2, 0x00020000);
    const int nsteps = (K + 127) >> 7;
    const int rot = start_step(walk.rot_stride, nsteps);
    struct Halves {
        Frag a[U][2], b[U][2][BT];
        uint32_t keep[U][2];
    } s0, s1;
    auto load = [&](Halves& st, int first) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int step = first + u * S;
            if (step < nsteps) { step += rot; step -= step >= nsteps ? nsteps : 0; }
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int at = step * 128 + hf * 32 + g * 8, k = at + sub * 64, kc = min(k, K - 8);
                st.keep[u][hf] = k < K ? 0xffffffffu : 0u;
                st.a[u][hf].u = *reinterpret_cast<const uint4*>(wrow + kc);
#pragma unroll
                for (int t = 0; t < BT; ++t) {  // a row past M lies outside the buffer's bounds: zeros, and no traffic
                    const int m = DIAG ? row : (t >> 1) * 16 + r, kx = DIAG ? kc : min(at + (t & 1) * 64, K - 8);
                    st.b[u][hf][t].i = __builtin_amdgcn_raw_buffer_load_b128(xres, (m * K + kx) * 2, 0, 0);
                }
            }
        }
    };
    f32x4_t acc[BT];
#pragma unroll
    for (int t = 0; t < BT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Halves& st) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                Frag a = st.a[u][hf];
                const uint32_t keep = st.keep[u][hf];
                a.u.x &= keep; a.u.y &= keep; a.u.z &= keep; a.u.w &= keep;
#pragma unroll
                for (int t = 0; t < BT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.v, st.b[u][hf][t].v, acc[t], 0, 0, 0);
            }
    };
    load(s0, wave);
    for (int step = wave; step < nsteps; step += 2 * U * S) {
        load(s1, step + U * S);
        __builtin_amdgcn_sched_barrier(0);
        multiply(s0);
        __builtin_amdgcn_sched_barrier(0);
        load(s0, step + 2 * U * S);
        __builtin_amdgcn_sched_barrier(0);
        multiply(s1);
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const f32x4_t first_half = acc[mt * (BT / MT)], second_half = acc[mt * (BT / MT) + BT / MT - 1];
        part[(wave * MT + mt) * 64 + lane] = g < 2 || DIAG ? first_half : second_half;
    }
    __syncthreads();
    halves_end<DIAG, OutT, TAIL>(p, tail, (const float*)part, MT * 256, S, M, n0, n1);
}

// The same through LDS (lds_stream.h): a step of 128 elements of K is two lines of each of the eight rows, and they lie in the slot
// as the tile's two halves; D steps are on their way.  The sums and their order are the kernel's above, which is left for rows that
// are too long for the buffers' 32-bit offsets, and for eight waves with more than sixteen rows of x, whose rings LDS cannot hold.
// Over cold weights, 8 / 16 / 32 / 64 rows of x, from registers -> here, us: 2,048 x 8,192 11.8 -> 8.6, 16.0 -> 10.4, 23.1 -> 13.7, 41.5 ->
// 21.5; 2,048 x 2,048 6.1 -> 4.6, 7.3 -> 5.0, 9.7 -> 6.1, 15.3 -> 9.0; 1,040 x 4,160 7.5 -> 5.2, 9.8 -> 6.0, 13.8 -> 8.1, 24.1 -> 11.5; 640 x
// 2,048 5.3 -> 3.9, 6.6 -> 4.3, 9.0 -> 5.4, 14.4 -> 7.3.  What bounds it: with few rows the start and the end (2.3 us for 300 x 72), then
// the weights (2,048 x 8,192: 3.9 TB/s); with many the reading of x, all of which every workgroup needs (64 rows of 8,192: 1 MB each).
template <int MT, bool DIAG, int D, typename OutT, bool TAIL>
__global__ __launch_bounds__(512) void gemm_skinny_halves_ring_kernel(const bf16_t* __restrict__ x_rows, const bf16_t* __restrict__ W, int M, int K, uint32_t items,
                                                                 uint32_t how, SkinnyProblem p, QkvTail tail) {
    static_assert(!DIAG || MT == 1, "both halves of K in a tile: eight rows of x");
    constexpr int BT = DIAG ? 1 : 2 * MT, SLOT = 2048 * (1 + BT), RING = D * SLOT, LOADS = 2 * (1 + BT), WAVE = RING / 16;
    extern __shared__ __attribute__((aligned(1024))) f32x4_t part[];  // the waves' rings, and then their sums, [64] each
    const Walk walk(how);
    const Share share = Share::of(items);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), S = walk.waves;
    const int r = lane & 15, g = lane >> 4, half = TAIL ? walk.d >> 1 : 1;
    const int n0 = share.begin(blockIdx.x), n1 = share.end(blockIdx.x);  // pairs, or rows
    const int nsteps = (K + 127) >> 7, rot = start_step(walk.rot_stride, nsteps);
    const int row = lane >> 3;  // the row that the lane's sixteen bytes are of
    int first = n0, at_row;     // of W: the row that the others are counted from, and the lane's
    if (TAIL) {
        const int pair = n0 + (row & 3);
        int e[2];
        tail_elements(walk, tail, pair % half, e);
        first = n0 / half * walk.d;
        at_row = pair < n1 ? pair / half * walk.d + (row < 4 ? e[0] : e[1]) - first : -1;
    } else {
        at_row = n0 + row < n1 ? row : -1;
    }
    const i32x4_t w = buffer_of(W + (long)first * K, (TAIL ? heads_of(n0, n1, half) * walk.d : n1 - n0) * K * 2);
    const i32x4_t x = buffer_of(x_rows, M * K * 2);
    const int w_at = at_row >= 0 ? at_row * K * 2 : LDS_PAST;
    int x_at[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) x_at[i] = row + 8 * i < M ? (row + 8 * i) * K * 2 : LDS_PAST;
    const int c8[2] = {stream_element(lane, 0), stream_element(lane, 1)};
    const char* ring = (const char*)(part + wave * WAVE);
    const unsigned to = __builtin_amdgcn_readfirstlane(lds_address(ring));
    auto issue = [&](int step, int slot) {
        int s = step + rot;
        s -= s >= nsteps ? nsteps : 0;
#pragma unroll
        for (int l = 0; l < LOADS; ++l) {  // W: a half of K a load; x: the same with eight rows, else a half of K a tile
            const int k = s * 128 + (l < 2 || DIAG ? l & 1 : (l - 2) >> 1 & 1) * 64 + c8[l & 1];
            const int from = l < 2 ? w_at : x_at[l < 2 || DIAG ? 0 : ((l - 2) >> 2) * 2 + (l & 1)];
            fetch16(l < 2 ? w : x, to + slot + l * 1024, from != LDS_PAST && k < K ? from + k * 2 : LDS_PAST);
        }
    };
    f32x4_t acc[BT];
#pragma unroll
    for (int t = 0; t < BT; ++t) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int in_row = r * 128 + ((g ^ (r >> 1)) & 7) * 16;
    bf16x8_t a[2], b[2][BT];
    auto read = [&](int slot) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const int at = (in_row ^ (hf * 64)) + slot;
            a[hf] = *reinterpret_cast<const bf16x8_t*>(ring + at);
#pragma unroll
            for (int t = 0; t < BT; ++t) b[hf][t] = *reinterpret_cast<const bf16x8_t*>(ring + at + 2048 * (1 + t));
        }
    };
    auto multiply = [&]() {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
            for (int t = 0; t < BT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[hf], b[hf][t], acc[t], 0, 0, 0);
    };
    const int n = wave < nsteps ? (nsteps - wave + S - 1) >> __builtin_ctz(S) : 0;  // the wave's steps
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < n) issue(wave + d * S, d * SLOT);
    int slot = 0, step = wave + D * S;
    for (int i = D; i < n; ++i, step += S) {
        wait_loads<(D - 1) * LOADS>();
        read(slot);
        wait_reads();
        __builtin_amdgcn_sched_barrier(0);
        issue(step, slot);  // into the slot just read
        __builtin_amdgcn_sched_barrier(0);
        multiply();
        slot = slot == RING - SLOT ? 0 : slot + SLOT;
    }
    RingTail<LOADS>::template last_steps<D - 1>(n, [&]() {
        read(slot);
        multiply();
        slot = slot == RING - SLOT ? 0 : slot + SLOT;
    });
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const f32x4_t first_half = acc[mt * (BT / MT)], second_half = acc[mt * (BT / MT) + BT / MT - 1];
        part[wave * WAVE + mt * 64 + lane] = g < 2 || DIAG ? first_half : second_half;
    }
    __syncthreads();
    halves_end<DIAG, OutT, TAIL>(p, tail, (const float*)part, WAVE * 4, S, M, n0, n1);
}

// The input product of a gated feed-forward, W = [gate rows, up rows], with the gate in its epilogue: y[M, F] = glu(x . Wg^T, x . Wu^T)
// for up to 16 rows.  A workgroup's two row tiles are the same rows of the gate and of the up matrix.  As a pass of its own
// the gate took 4.5 us behind a product of 13 (2 rows, 2 x 5,504 x 2,048).
template <int D>
__global__ __launch_bounds__(512) void gemm_skinny_glu_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, int M, int F, int K,
                                                              uint32_t items, uint32_t how, bf16_t* __restrict__ y, int kind, float alpha, float limit) {
    extern __shared__ __attribute__((aligned(1024))) f32x4_t part[];  // the waves' rings, and then their sums, [2][64] each
    constexpr int WAVE = D == 0 ? 128 : RowStream<2, D == 0 ? 1 : D>::RING / 16;
    const Walk walk(how);
    const Share share = Share::of(items);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, S = walk.waves;
    const int n0 = share.begin(blockIdx.x), n1 = share.end(blockIdx.x);
    const int nsteps = (K + 63) >> 6, rot = start_step(walk.rot_stride, nsteps);
    f32x4_t acc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
    if constexpr (D > 0) {
        RowStream<2, D> rows;
        rows.w[0] = buffer_of(W + (long)n0 * K, (n1 - n0) * K * 2);
        rows.w[1] = buffer_of(W + (long)(F + n0) * K, (n1 - n0) * K * 2);
        rows.x = buffer_of(x, M * K * 2);
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            const int i = stream_row(lane, l);
            rows.w_at[l] = rows.w_at[2 + l] = i < n1 - n0 ? i * K * 2 : LDS_PAST;
            rows.x_at[l] = i < M ? i * K * 2 : LDS_PAST;
        }
        rows.run(acc, (const char*)(part + wave * WAVE), lane, wave, S, K, nsteps, rot);
    } else {
        const int row = min(n0 + (lane & 15), n1 - 1);
        const bf16_t* wrow[2] = {W + (long)row * K, W + (long)(F + row) * K};
        f32x4_t sums[2][1] = {{acc[0]}, {acc[1]}};
        by_registers<1, 2, 2>(sums, wrow, x, lane, wave, S, M, K, nsteps, rot);
        acc[0] = sums[0][0], acc[1] = sums[1][0];
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) part[wave * WAVE + rt * 64 + lane] = acc[rt];
    __syncthreads();
    const float* sums = (const float*)part;  // feature i of a tile, row m of x: lane (i / 4) * 16 + m, element i % 4
    for (int item = threadIdx.x; item < 16 * M; item += S * 64) {
        const int m = item >> 4, i = item & 15;
        if (n0 + i >= n1) continue;
        const int at = ((i >> 2) * 16 + m) * 4 + (i & 3);
        float gate = sums[at], up = sums[256 + at];
        for (int w = 1; w < S; ++w) gate += sums[w * WAVE * 4 + at], up += sums[w * WAVE * 4 + 256 + at];
        y[(long)m * F + n0 + i] = f32_to_bf16_bits(glu_value(kind, round_to_bf16(gate), round_to_bf16(up), alpha, limit));
    }
}

// The product of few rows together with the LayerNorm in front of it, y = act(LN(x) . W^T + bias), rows of up to 2,048
// elements.  As launches of their own a norm of a few rows takes 4.7 us, nearly all of it what any launch costs; here every
// workgroup norms the rows for itself while its rows of W are on their way: rows of x are asked for first, then the norm's
// vectors, then all of the workgroup's W (a range of up to 2,048 elements: 16 loads a lane), so that the norm waits for its own
// loads alone.  Normed rows lie in LDS, rounded to bfloat16 as the norm's own launch stores them, and are read from there as the
// B operand: x passes the address path once a workgroup, not once a wave.  Statistics in 32-bit, mean first.
// TAIL: a fused query_key_value product taken to its end as by gemm_skinny_tail_kernel.
// Sizes of W alone choose the waves and with them the order of summation: eight, which finish the norm sooner, up to a workgroup
// a compute unit and a sixteenth, else four, which leave room for a second one (8,192 x 2,048 at 5 rows: 12.4 and 11.7 us).  A wave
// norms up to four rows then, two at a time (of 2,048 elements one), so that the registers do not run out.
// Replays over cold weights, norm and product (GELU) -> this, 5 / 8 / 9 / 16 rows: 3,120 x 1,040 9.0 -> 5.1, 9.1 -> 5.2, 9.1 -> 5.7, 9.2
// -> 6.1; 4,160 x 1,040 9.4 -> 6.3, 9.7 -> 6.8, 9.8 -> 8.7, 10.0 -> 9.4; 6,144 x 1,536 12.6 -> 8.5, 12.8 -> 8.8, 12.9 -> 10.8, 13.6 -> 11.4;
// 8,192 x 2,048 16.2 -> 11.9, 16.4 -> 12.0, 15.8 -> 15.2, 16.8 -> 16.3.
template <int NORMED_WAVES, int CH, int RW, bool TAIL>  // CH: groups of 512 elements of a row; RW: rows of x a wave norms
__global__ __launch_bounds__(NORMED_WAVES * 64, RW == 4 ? 2 : 1) void gemm_normed_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ W, const float* __restrict__ ln_w, const float* __restrict__ ln_b, int M, int K, uint32_t items,
    uint32_t how, float eps, SkinnyProblem p, QkvTail tail) {
    constexpr int STEPS = 8 * CH / NORMED_WAVES;  // steps of 64 elements of K a wave takes
    extern __shared__ f32x4_t part[];  // [waves][64], then the normed rows [M][K + 8]
    bf16_t* rows = (bf16_t*)(part + NORMED_WAVES * 64);
    const int pitch = K + 8;  // sixteen bytes between rows keep the reads of sixteen rows on distinct banks
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const Walk walk(how);
    const Share share = Share::of(items);
    const int r = lane & 15, g = lane >> 4, half = TAIL ? walk.d >> 1 : 1;
    const int n0 = share.begin(blockIdx.x), n1 = share.end(blockIdx.x);
    const int chunks = K >> 3;
    constexpr int RB = RW < 2 || (RW == 4 && CH == 4) ? 1 : 2;  // rows normed at a time: what leaves registers for two workgroups of four waves a unit
    uint4 xv[RB][CH];
    float gain[CH][8], shift[CH][8];
    auto load_rows = [&](int b) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < CH; ++j)
                xv[i][j] = *reinterpret_cast<const uint4*>(x + (long)min(wave + (b + i) * NORMED_WAVES, M - 1) * K + min(lane + j * 64, chunks - 1) * 8);
    };
    load_rows(0);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const int at = min(lane + j * 64, chunks - 1) * 8;
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            *reinterpret_cast<float4*>(&gain[j][e]) = *reinterpret_cast<const float4*>(ln_w + at + e);
            *reinterpret_cast<float4*>(&shift[j][e]) = *reinterpret_cast<const float4*>(ln_b + at + e);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    int w_row = min(n0 + r, n1 - 1);
    if (TAIL) {  // as in gemm_skinny_tail_kernel
        const int mine = min(n0 + (r & 7), n1 - 1);
        int e[2];
        tail_elements(walk, tail, mine % half, e);
        w_row = mine / half * walk.d + (r < 8 ? e[0] : e[1]);
    }
    const bf16_t* wrow = W + (long)w_row * K;
    Frag a[STEPS][2];
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
            a[u][hf].u = *reinterpret_cast<const uint4*>(wrow + min((wave + u * NORMED_WAVES) * 64 + hf * 32 + g * 8, K - 8));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < RW; b += RB) {
        float v[RB][CH][8], sum[RB], mean[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            sum[i] = 0.f;
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                unpack8(xv[i][j], v[i][j]);
#pragma unroll
                for (int e = 0; e < 8; ++e) sum[i] += lane + j * 64 < chunks ? v[i][j][e] : 0.f;
            }
        }
        if (b + RB < RW) {  // the next rows, which come behind W, while these are normed
            load_rows(b + RB);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) sum[i] = wave_sum(sum[i]);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            mean[i] = sum[i] / (float)K;
            sum[i] = 0.f;
#pragma unroll
            for (int j = 0; j < CH; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    v[i][j][e] -= mean[i];
                    sum[i] += lane + j * 64 < chunks ? v[i][j][e] * v[i][j][e] : 0.f;
                }
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) sum[i] = wave_sum(sum[i]);
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const int m = wave + (b + i) * NORMED_WAVES;
            if (m >= M) break;
            const float rstd = 1.0f / sqrtf(sum[i] / (float)K + eps);
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                float o[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = v[i][j][e] * rstd * gain[j][e] + shift[j][e];
                if (lane + j * 64 < chunks) *reinterpret_cast<uint4*>(rows + m * pitch + (lane + j * 64) * 8) = pack8(o);
            }
        }
    }
    // the barrier waits for LDS alone: W stays on its way
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const bf16_t* mine = rows + min(r, M - 1) * pitch;  // (columns past M repeat the last row and are not stored)
#pragma unroll
    for (int u = 0; u < STEPS; ++u)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const int k = (wave + u * NORMED_WAVES) * 64 + hf * 32 + g * 8;
            const uint32_t keep = k < K ? 0xffffffffu : 0u;
            Frag b;
            b.u = *reinterpret_cast<const uint4*>(mine + min(k, K - 8));
            a[u][hf].u.x &= keep; a[u][hf].u.y &= keep; a[u][hf].u.z &= keep; a[u][hf].u.w &= keep;
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][hf].v, b.v, acc, 0, 0, 0);
        }
    part[wave * 64 + lane] = acc;
    __syncthreads();
    const float* sums = (const float*)part;  // row i of the tile, column m: lane (i / 4) * 16 + m, element i % 4
    auto sum_of = [&](int m, int i) {
        const int at = ((i >> 2) * 16 + m) * 4 + (i & 3);
        float s = sums[at];
#pragma unroll
        for (int w = 1; w < NORMED_WAVES; ++w) s += sums[w * 256 + at];
        return s;
    };
    const int per = TAIL ? 8 : 16;
    for (int item = threadIdx.x; item < per * M; item += NORMED_WAVES * 64) {
        const int m = item / per, i = item % per, n = n0 + i;
        if (n >= n1) continue;
        if constexpr (TAIL) qkv_tail_pair(tail, p.bias, m, n / half, n % half, round_to_bf16(sum_of(m, i)), round_to_bf16(sum_of(m, i + 8)));
        else store_feature<bf16_t>((bf16_t*)p.y, p.bias, p.act, nullptr, nullptr, p.N, m, n, sum_of(m, i));
    }
}

// Waves per workgroup, i.e. how many ways K is split, by the sizes of W alone, never by M or by the tile variant, so the order of
// summation is the same for every batch.  Long streams per wave beat many short ones, so K is split where N alone gives too
// few waves, and where rows are long (each wave then walks fewer rows' pages at a time).  Measured over cold weights, us with 1 / 2 / 4
// waves, 8 rows of x, by tiles of 32 rows of W: 41,984 x 8,192 129 / 127 / 124, 65,024 x 4,544 108 / 110 / 112, 22,848 x 4,544 42.0 / 39.7 /
// 43.1, 22,528 x 4,096 36.2 / 35.6 / 38.7, 32,768 x 2,048 26.6 / 28.6 / 32.5, 8,192 x 2,048 11.2 / 8.5 / 8.9, 6,144 x 2,048 11.1 / 7.5 / 7.8; by
// tiles of sixteen 12,032 x 8,192 38.1 / 39.5 / 37.3, 12,032 x 4,096 20.5 / 21.4 / 21.6, 11,008 x 2,048 11.0 / 11.7 / 12.6.
static int pick_split(int N, int K) {
    if (N >= 10240 && K >= 8192) return 4;
    if (N >= 32768 || (N >= 10240 && N < 16384)) return 1;
    if (N >= 16384) return K >= 4096 ? 2 : 1;
    if (N >= 4096) return 2;
    if (N >= 1024) return 4;
    return 8;
}

// Whether up to sixteen rows of x go by tiles of sixteen rows of W a wave (else of 32, which read x half as often; the bits are the
// same): where 32 leave compute units with an uneven share, and for short rows, whose waves spend their time starting.  32 rows -> 16, us:
// 11,008 x 2,048 12.0 -> 11.0, 12,032 x 8,192 42.0 -> 37.3; 50,001 x 1,040 1 row 28.5 -> 22.5, 8 rows 28.8 -> 26.6, 16 rows 31.0 -> 31.2.
static bool short_tiles(int N, int K, int M) { return (N >= 10240 && N < 16384) || (N >= 16384 && K <= 2048 && M <= 8); }

// One launch of a kernel whose waves each have a ring in LDS (D > 0): more than 64 KB have to be asked for, on every device
template <typename Kernel, typename... Args>
static int launch_rings(Kernel kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s, Args... args) {
    if (lds > 64 * 1024 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return pta_fail("gemm_skinny_bf16: %zu bytes of LDS were refused", lds);
    hipLaunchKernelGGL(kernel, grid, block, lds, s, args...);
    return 0;
}

// gemm_skinny_kernel, in the order that it takes its arguments in
template <typename Kernel>
static int launch_two(Kernel kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s, const SkinnyProblem& a, const SkinnyProblem& b, int M, int K, int rot_stride,
                      const QkvTail& tail = QkvTail{}) {
    PTA_REQUIRE(a.rows.fits() && b.rows.fits(), "gemm_skinny_bf16: %d workgroups are too many for one launch", (int)grid.x);
    return launch_rings(kernel, grid, block, lds, s, a.x, a.W, b.x, b.W, M, K, a.blocks, a.rows.packed(), b.rows.packed(),
                        Walk::packed((int)block.x / 64, rot_stride, tail.d), a, b, tail);
}

template <int MT, int RT, int U, typename OutT>
static int launch_cfg(SkinnyProblem a, SkinnyProblem b, int M, int K, int S, hipStream_t s, bool spread = false) {
    const int rows = 16 * RT;
    if (S <= 0) S = pick_split(a.N + b.N, K);
    a.blocks = (a.N + rows - 1) / rows;
    b.blocks = (b.N + rows - 1) / rows;
    // A launch takes as long as the compute unit with the most workgroups: 714 workgroups on 256 units take
    // the time of 768 (measured: 44.7 us for 22,848 rows, 45.5 us for 24,576).  So a launch with more
    // workgroups than units gets a whole number of workgroups per unit, each with a little fewer rows.
    const int units = pta_compute_units(), natural = a.blocks + b.blocks;
    if (spread) {
        a.blocks = std::max(a.blocks, std::min(units, (a.N + 3) / 4));
    } else if (natural > units && natural % units != 0) {
        const int total = (natural + units - 1) / units * units;
        if (b.blocks == 0) {
            a.blocks = total;
        } else {
            const int first = (int)((long)total * a.N / (a.N + b.N));
            a.blocks = std::max(a.blocks, std::min(first, total - b.blocks));
            b.blocks = total - a.blocks;
        }
    }
    a.rows = Share(a.N, a.blocks);
    b.rows = Share(b.N, b.blocks);
    const dim3 grid(a.blocks + b.blocks), block(S * 64);
    const size_t lds = (size_t)S * RT * MT * 64 * sizeof(f32x4_t);
    static const int rot_env = getenv("PTA_SKINNY_ROT") ? atoi(getenv("PTA_SKINNY_ROT")) : -1;
    const int rot_stride = rot_env >= 0 ? rot_env : (K % 2048 == 0 ? 5 : 0);  // rows a multiple of 4 KB long
    if constexpr (MT == 1 && RT <= 2) if (K <= STREAM_MOST_K) {
        if (S <= 4) return launch_two(gemm_skinny_kernel<MT, RT, U, OutT, 0, 4>, grid, block, (size_t)S * RowStream<RT, 4>::RING, s, a, b, M, K, rot_stride);
        return launch_two(gemm_skinny_kernel<MT, RT, U, OutT, 0, 3>, grid, block, (size_t)S * RowStream<RT, 3>::RING, s, a, b, M, K, rot_stride);
    }
    return launch_two(gemm_skinny_kernel<MT, RT, U, OutT>, grid, block, lds, s, a, b, M, K, rot_stride);
}

// where a workgroup has eight rows of W or fewer (N alone decides: one order of summation for any number of rows of x)
static bool by_halves(int N) { return N <= 8 * pta_compute_units(); }

template <int N> using I = std::integral_constant<int, N>;

template <typename OutT, bool TAIL = false>
static int launch_halves(SkinnyProblem p, int M, int K, int S, hipStream_t s, const QkvTail& tail = QkvTail{}) {
    const int items = TAIL ? p.N / 2 : p.N, most = TAIL ? 4 : 8, units = pta_compute_units();
    // Waves by N alone, as the order of the sums must not depend on x: four where a workgroup has five rows or fewer and its waves
    // spend their time starting (8 rows of x, two -> four: 1,040 x 4,160 5.2 -> 4.9 us, 640 x 2,048 3.6 -> 3.2, 1,024 x 4,096 5.1 -> 4.8),
    // else two (2,048 x 8,192 8.3, four 9.0; 2,048 x 2,048 4.3, four 4.6).
    if (S <= 0) S = p.N <= 5 * units ? 4 : 2;
    const dim3 grid(std::max((items + most - 1) / most, std::min(units, (items + most / 2 - 1) / (most / 2)))), block(S * 64);
    p.rows = Share(items, (int)grid.x);
    PTA_REQUIRE(p.rows.fits(), "gemm_skinny_bf16: %d workgroups are too many for one launch", (int)grid.x);
    static const int rot_env = getenv("PTA_SKINNY_ROT") ? atoi(getenv("PTA_SKINNY_ROT")) : -1;
    const int rot = rot_env >= 0 ? rot_env : (K % 2048 == 0 ? 3 : 0);
    const uint32_t how = Walk::packed(S, rot, tail.d, TAIL && qkv_tail_plain_pairs(tail.rot, tail.d));
    auto go = [&](auto kernel, int tiles) { hipLaunchKernelGGL(kernel, grid, block, (size_t)S * tiles * 64 * sizeof(f32x4_t), s, p.x, p.W, M, K, p.rows.packed(), how, p, tail); };
    if (K <= STREAM_MOST_K && (M <= 16 || S <= 4)) {
        int rc = 0;
        auto ring = [&](auto kernel, int bytes) { rc = launch_rings(kernel, grid, block, (size_t)S * bytes, s, p.x, p.W, M, K, p.rows.packed(), how, p, tail); };
        auto of_depth = [&](auto tiles, auto few, auto two, auto four, auto eight) {  // loads on their way that LDS has room for
            constexpr int MT = tiles(), SLOT = 2048 * (few() ? 2 : 1 + 2 * MT);
            if (S <= 2) ring(gemm_skinny_halves_ring_kernel<MT, few(), two(), OutT, TAIL>, two() * SLOT);
            else if (S <= 4) ring(gemm_skinny_halves_ring_kernel<MT, few(), four(), OutT, TAIL>, four() * SLOT);
            else if constexpr (eight() > 0) ring(gemm_skinny_halves_ring_kernel<MT, few(), eight(), OutT, TAIL>, eight() * SLOT);
        };
        if (M <= 8) of_depth(I<1>(), std::true_type(), I<6>(), I<6>(), I<4>());
        else if (M <= 16) of_depth(I<1>(), std::false_type(), I<6>(), I<6>(), I<3>());
        else if constexpr (!TAIL) {
            if (M <= 32) of_depth(I<2>(), std::false_type(), I<4>(), I<3>(), I<0>());
            else if (M <= 48) of_depth(I<3>(), std::false_type(), I<4>(), I<2>(), I<0>());
            else of_depth(I<4>(), std::false_type(), I<4>(), I<2>(), I<0>());
        }
        return rc ? rc : pta_check_launch("gemm_skinny_bf16");
    }
    if (M <= 8) go(gemm_skinny_halves_kernel<1, true, 2, OutT, TAIL>, 1);
    else if (M <= 16) go(gemm_skinny_halves_kernel<1, false, 2, OutT, TAIL>, 1);
    else if constexpr (!TAIL) {
        if (M <= 32) go(gemm_skinny_halves_kernel<2, false, 1, OutT, false>, 2);
        else if (M <= 48) go(gemm_skinny_halves_kernel<3, false, 1, OutT, false>, 3);
        else go(gemm_skinny_halves_kernel<4, false, 1, OutT, false>, 4);
    }
    return pta_check_launch("gemm_skinny_bf16");
}

template <typename OutT>
static int launch_skinny(SkinnyProblem a, SkinnyProblem b, int M, int K, int variant, int S, hipStream_t s) {
    // variant: row tiles per wave and steps per stage (6: one tile, its rows spread over all units; 7: eight rows at two places of
    // K); 0: chosen here
    // Tiles of 32 rows of W that would occupy half of the compute units or fewer: a unit pulls no more than some 24 GB/s, so
    // the rows are spread over all units instead, a few rows each (the rest of a tile's lanes read a row again).  Replays over
    // cold weights, 8 rows of x, 32-row tiles -> spread: 3,072 x 2,048 9.8 -> 7.0 us (up to eight rows a unit:
    // gemm_skinny_halves_kernel); with more tiles the second read of x costs more than the units win (5,504
    // x 2,048 9.2 -> 9.8, at 16 rows of x 9.9 -> 11.7).
    if (variant == 7 || (variant == 0 && b.N == 0 && by_halves(a.N))) return launch_halves<OutT>(a, M, K, S, s);
    if (variant == 0 && b.N == 0 && pta_gemm_skinny_spread(a.N)) variant = 6;
    int rc;
    if (M <= 16) {
        if (variant == 0) variant = short_tiles(a.N + b.N, K, M) ? 1 : 2;
        if (variant == 1) rc = launch_cfg<1, 1, 4, OutT>(a, b, M, K, S, s);
        else if (variant == 2) rc = launch_cfg<1, 2, 2, OutT>(a, b, M, K, S, s);
        else if (variant == 3) rc = launch_cfg<1, 4, 1, OutT>(a, b, M, K, S, s);
        else if (variant == 4) rc = launch_cfg<1, 4, 2, OutT>(a, b, M, K, S, s);
        else if (variant == 6) rc = launch_cfg<1, 1, 2, OutT>(a, b, M, K, S, s, true);
        else rc = launch_cfg<1, 2, 4, OutT>(a, b, M, K, S, s);
    } else if (M <= 32) {
        if (variant == 3 || variant == 4) rc = launch_cfg<2, 4, 1, OutT>(a, b, M, K, S, s);
        else if (variant == 6) rc = launch_cfg<2, 1, 1, OutT>(a, b, M, K, S, s, true);
        else rc = launch_cfg<2, 2, 1, OutT>(a, b, M, K, S, s);
    } else if (M <= 48) {
        if (variant == 6) rc = launch_cfg<3, 1, 1, OutT>(a, b, M, K, S, s, true);
        else rc = launch_cfg<3, 2, 1, OutT>(a, b, M, K, S, s);
    } else {
        if (variant == 3 || variant == 4) rc = launch_cfg<4, 4, 1, OutT>(a, b, M, K, S, s);
        else if (variant == 6) rc = launch_cfg<4, 1, 1, OutT>(a, b, M, K, S, s, true);
        else rc = launch_cfg<4, 2, 1, OutT>(a, b, M, K, S, s);
    }
    if (rc) return rc;
    return pta_check_launch("gemm_skinny_bf16");
}

static bool in_kernel(int act) { return act == PTA_ACT_NONE || act == PTA_ACT_GELU || act == PTA_ACT_RELU2; }

static int check_skinny(const char* what, const void* y, const void* x, const void* W, int M, int N, int K, int act) {
    PTA_REQUIRE(M > 0 && N > 0 && K > 0, "%s: sizes must be positive (M=%d N=%d K=%d)", what, M, N, K);
    PTA_REQUIRE(M <= 64, "%s: at most 64 rows, got %d (use the library product)", what, M);
    PTA_REQUIRE(K % 8 == 0, "%s: K=%d must be a multiple of 8 (16-byte loads)", what, K);
    PTA_REQUIRE(y && x && W, "%s: null pointer", what);
    PTA_REQUIRE((long)M * K * 2 < (1L << 31), "%s: x is too large for 32-bit buffer offsets", what);
    PTA_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)W % 16) == 0, "%s: x and W must be 16-byte aligned", what);
    PTA_REQUIRE(pta_act_known(act), "%s: unknown activation %d", what, act);
    return 0;
}

extern "C" int pta_gemm_skinny_bf16(void* y, const void* x, const void* W, const float* bias, const void* add1,
                                    const void* add2, int M, int N, int K, int act, int out_f32, int variant,
                                    int waves, void* stream) {
    if (check_skinny("gemm_skinny_bf16", y, x, W, M, N, K, act)) return 1;
    PTA_REQUIRE(variant >= 0 && variant <= 7, "gemm_skinny_bf16: unknown variant %d", variant);
    PTA_REQUIRE(waves == 0 || (waves >= 1 && waves <= 8 && (waves & (waves - 1)) == 0),
                "gemm_skinny_bf16: waves per workgroup must be 0 (choose) or a power of two up to 8, got %d", waves);
    hipStream_t s = (hipStream_t)stream;
    const SkinnyProblem none{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0, 0};
    PTA_REQUIRE(!out_f32 || act == PTA_ACT_NONE || act == PTA_ACT_GELU, "gemm_skinny_bf16: activation %d needs a bfloat16 result", act);
    if (!in_kernel(act)) {
        // the kernel's epilogue knows the exact GELU and the squared ReLU only (every activation there would cost it its
        // unrolled loops): the product with its bias first, then activation and additions as a pass over y
        const SkinnyProblem plain{y, (const bf16_t*)x, (const bf16_t*)W, bias, nullptr, nullptr, N, PTA_ACT_NONE, 0};
        if (launch_skinny<bf16_t>(plain, none, M, K, variant, waves, s)) return 1;
        return pta_epilogue(y, N, nullptr, add1, add2, M, N, act, PTA_BF16, stream);
    }
    const SkinnyProblem a{y, (const bf16_t*)x, (const bf16_t*)W, bias, (const bf16_t*)add1, (const bf16_t*)add2, N, act, 0};
    if (out_f32) return launch_skinny<float>(a, none, M, K, variant, waves, s);
    return launch_skinny<bf16_t>(a, none, M, K, variant, waves, s);
}

// The pair launch of a decode step whose first product is a fused query_key_value projection: its rows never
// reach memory as such; queries come out rotated in q_out [M, heads, d], keys (rotated) and values go to the
// cache pages of their sequences, as pta_qkv_rope_cache would have left them.  Up to 16 rows, head sizes that are
// multiples of 32.  The second product is y2 = act2(x2 . W2^T + bias2) as in the plain pair.
extern "C" int pta_gemm_skinny_pair_qkv_bf16(void* q_out, const void* x1, const void* W1, const float* bias1,
                                             const PtaRotation* rotation, const int* token_pos,
                                             const int* token_seq, const int* block_table, int bt_stride, void* k_pool,
                                             void* v_pool, int nh, int nkv, int d, int layout, int write_cache, void* y2,
                                             const void* x2, const void* W2, const float* bias2, int N2, int act2, int M,
                                             int K, void* stream) {
    PTA_REQUIRE(nh > 0 && nkv > 0 && d > 0 && nh % nkv == 0, "gemm_skinny_pair_qkv_bf16: heads %d, kv heads %d, head size %d", nh, nkv, d);
    const int N1 = (nh + 2 * nkv) * d;
    if (check_skinny("gemm_skinny_pair_qkv_bf16", q_out, x1, W1, M, N1, K, PTA_ACT_NONE)) return 1;
    if (check_skinny("gemm_skinny_pair_qkv_bf16", y2, x2, W2, M, N2, K, act2)) return 1;
    PTA_REQUIRE(M <= 16, "gemm_skinny_pair_qkv_bf16: at most 16 rows, got %d", M);
    PTA_REQUIRE(d % 32 == 0 && d <= 256, "gemm_skinny_pair_qkv_bf16: head size %d must be a multiple of 32 up to 256", d);
    PTA_REQUIRE(layout >= 0 && layout <= 2, "gemm_skinny_pair_qkv_bf16: unknown layout %d", layout);
    PTA_REQUIRE(layout != PTA_QKV_TAIL || nkv == 1, "gemm_skinny_pair_qkv_bf16: the tail layout has one kv head, got %d", nkv);
    PTA_REQUIRE(layout != PTA_QKV_INTERLEAVED || nkv == nh, "gemm_skinny_pair_qkv_bf16: the interleaved layout needs kv heads == heads");
    PTA_REQUIRE(token_pos, "gemm_skinny_pair_qkv_bf16: null token positions");
    const PtaRotation rot = pta_rotation_of(rotation);
    if (pta_check_rotation("gemm_skinny_pair_qkv_bf16", rot, d, token_seq)) return 1;
    PTA_REQUIRE(!write_cache || (k_pool && v_pool && block_table && token_seq), "gemm_skinny_pair_qkv_bf16: null cache pointer");
    PTA_REQUIRE((((uintptr_t)q_out | (uintptr_t)k_pool) % 8) == 0, "gemm_skinny_pair_qkv_bf16: outputs must be 8-byte aligned");
    SkinnyProblem a{nullptr, (const bf16_t*)x1, (const bf16_t*)W1, bias1, nullptr, nullptr, N1, PTA_ACT_NONE, 0};
    SkinnyProblem b{y2, (const bf16_t*)x2, (const bf16_t*)W2, bias2, nullptr, nullptr, N2, in_kernel(act2) ? act2 : 0, 0};
    const QkvTail tail{(bf16_t*)q_out, rot, token_pos, token_seq, block_table, bt_stride, (bf16_t*)k_pool,
                       (bf16_t*)v_pool, nh, nkv, d, layout, write_cache};
    // the first product's workgroups are bound to heads; the second one's fill the launch up to a whole number per unit
    a.blocks = (nh + 2 * nkv) * (d / 32);
    b.blocks = (N2 + 31) / 32;
    const int units = pta_compute_units(), natural = a.blocks + b.blocks;
    if (natural > units && natural % units != 0) b.blocks = (natural + units - 1) / units * units - a.blocks;
    a.rows = Share(a.N, a.blocks);
    b.rows = Share(b.N, b.blocks);
    const int S = pick_split(N1 + N2, K);
    static const int rot_env = getenv("PTA_SKINNY_ROT") ? atoi(getenv("PTA_SKINNY_ROT")) : -1;
    const int rot_stride = rot_env >= 0 ? rot_env : (K % 2048 == 0 ? 5 : 0);
    auto go = [&](auto kernel, size_t ring) {
        return launch_two(kernel, dim3(a.blocks + b.blocks), dim3(S * 64), S * ring, (hipStream_t)stream, a, b, M, K, rot_stride, tail);
    };
    const bool plain = qkv_tail_plain_pairs(rot, d);
    int rc;
    if (K > STREAM_MOST_K) rc = plain ? go(gemm_skinny_kernel<1, 2, 2, bf16_t, 1>, 2048) : go(gemm_skinny_kernel<1, 2, 2, bf16_t, 2>, 2048);
    else if (S <= 4) rc = plain ? go(gemm_skinny_kernel<1, 2, 2, bf16_t, 1, 4>, RowStream<2, 4>::RING) : go(gemm_skinny_kernel<1, 2, 2, bf16_t, 2, 4>, RowStream<2, 4>::RING);
    else rc = plain ? go(gemm_skinny_kernel<1, 2, 2, bf16_t, 1, 3>, RowStream<2, 3>::RING) : go(gemm_skinny_kernel<1, 2, 2, bf16_t, 2, 3>, RowStream<2, 3>::RING);
    if (rc) return rc;
    if (pta_check_launch("gemm_skinny_pair_qkv_bf16")) return 1;
    if (!in_kernel(act2)) return pta_epilogue(y2, N2, nullptr, nullptr, nullptr, M, N2, act2, PTA_BF16, stream);
    return 0;
}

// Whether pta_gemm_skinny_qkv_bf16 is the launch for a fused product of so many rows of W: where they are spread over the units
extern "C" int pta_gemm_skinny_spread(int N) { return N > 0 && (N + 31) / 32 <= pta_compute_units() / 2; }

// The operands of a fused query_key_value projection on its own, checked: up to 16 rows, any even head size up to 256
static int make_tail_problem(const char* what, void* q_out, const void* x, const void* W, const float* bias, const PtaRotation* rotation,
                             const int* token_pos, const int* token_seq, const int* block_table, int bt_stride, void* k_pool, void* v_pool,
                             int nh, int nkv, int d, int layout, int write_cache, int M, int K, SkinnyProblem& p, QkvTail& tail) {
    PTA_REQUIRE(nh > 0 && nkv > 0 && d > 0 && nh % nkv == 0, "%s: heads %d, kv heads %d, head size %d", what, nh, nkv, d);
    const int N = (nh + 2 * nkv) * d;
    if (check_skinny(what, q_out, x, W, M, N, K, PTA_ACT_NONE)) return 1;
    PTA_REQUIRE(M <= 16, "%s: at most 16 rows, got %d", what, M);
    PTA_REQUIRE(d % 2 == 0 && d <= 256, "%s: head size %d must be even and at most 256", what, d);
    PTA_REQUIRE(layout >= 0 && layout <= 2, "%s: unknown layout %d", what, layout);
    PTA_REQUIRE(layout != PTA_QKV_TAIL || nkv == 1, "%s: the tail layout has one kv head, got %d", what, nkv);
    PTA_REQUIRE(layout != PTA_QKV_INTERLEAVED || nkv == nh, "%s: the interleaved layout needs kv heads == heads", what);
    PTA_REQUIRE(token_pos, "%s: null token positions", what);
    const PtaRotation rot = pta_rotation_of(rotation);
    if (pta_check_rotation(what, rot, d, token_seq)) return 1;
    PTA_REQUIRE(!write_cache || (k_pool && v_pool && block_table && token_seq), "%s: null cache pointer", what);
    p = SkinnyProblem{nullptr, (const bf16_t*)x, (const bf16_t*)W, bias, nullptr, nullptr, N, PTA_ACT_NONE, 0};
    tail = QkvTail{(bf16_t*)q_out, rot, token_pos, token_seq, block_table, bt_stride, (bf16_t*)k_pool,
                   (bf16_t*)v_pool, nh, nkv, d, layout, write_cache};
    return 0;
}

// A fused query_key_value projection on its own for up to 16 rows, with the tail of pta_gemm_skinny_pair_qkv_bf16; any even
// head size up to 256, N = (nh + 2 nkv) d within pta_gemm_skinny_spread.
extern "C" int pta_gemm_skinny_qkv_bf16(void* q_out, const void* x, const void* W, const float* bias, const PtaRotation* rotation,
                                        const int* token_pos, const int* token_seq, const int* block_table, int bt_stride,
                                        void* k_pool, void* v_pool, int nh, int nkv, int d, int layout, int write_cache, int M, int K,
                                        void* stream) {
    SkinnyProblem p;
    QkvTail tail;
    if (make_tail_problem("gemm_skinny_qkv_bf16", q_out, x, W, bias, rotation, token_pos, token_seq, block_table, bt_stride, k_pool,
                          v_pool, nh, nkv, d, layout, write_cache, M, K, p, tail)) return 1;
    const int N = p.N;
    PTA_REQUIRE(pta_gemm_skinny_spread(N), "gemm_skinny_qkv_bf16: %d rows of W are too many for this launch", N);
    if (by_halves(N)) return launch_halves<bf16_t, true>(p, M, K, 0, (hipStream_t)stream, tail);
    const int pairs = N / 2;
    const int blocks = std::max((pairs + 7) / 8, std::min(pta_compute_units(), (pairs + 1) / 2));
    const int S = pick_split(N, K);
    static const int rot_env = getenv("PTA_SKINNY_ROT") ? atoi(getenv("PTA_SKINNY_ROT")) : -1;
    const int rot_stride = rot_env >= 0 ? rot_env : (K % 2048 == 0 ? 5 : 0);
    auto go = [&](auto kernel, size_t ring) {
        return launch_rings(kernel, dim3(blocks), dim3(S * 64), S * ring, (hipStream_t)stream, p.x, p.W, M, K, Share(pairs, blocks).packed(),
                            Walk::packed(S, rot_stride, d, qkv_tail_plain_pairs(tail.rot, d)), bias, tail);
    };
    if (K > STREAM_MOST_K ? go(gemm_skinny_tail_kernel<0>, 1024) : go(gemm_skinny_tail_kernel<4>, RowStream<1, 4>::RING)) return 1;
    return pta_check_launch("gemm_skinny_qkv_bf16");
}

// Whether the two entry points below take so many rows of x, elements of K and rows of W: each workgroup norms the rows again, which
// pays with up to two workgroups a compute unit.  One answer for up to sixteen rows of x: a batch's size changes no bit of a sequence
extern "C" int pta_gemm_normed_ok(int M, int N, int K) {
    return M > 0 && M <= 16 && K > 0 && K % 8 == 0 && K <= 2048 && N > 0 && N <= 32 * pta_compute_units();
}

template <bool TAIL>
static int launch_normed(const char* what, SkinnyProblem p, const float* ln_w, const float* ln_b, float eps, int M, int K,
                         const QkvTail& tail, hipStream_t s) {
    PTA_REQUIRE(pta_gemm_normed_ok(M, p.N, K), "%s: M=%d N=%d K=%d are not for this launch", what, M, p.N, K);
    PTA_REQUIRE(ln_w && ln_b && ((uintptr_t)ln_w % 16) == 0 && ((uintptr_t)ln_b % 16) == 0, "%s: the norm's vectors must be there and 16-byte aligned", what);
    const int items = TAIL ? p.N / 2 : p.N, most = TAIL ? 8 : 16, units = pta_compute_units();
    const int groups = std::max((items + most - 1) / most, std::min(units, (items + most / 4 - 1) / (most / 4)));
    p.rows = Share(items, groups);
    PTA_REQUIRE(p.rows.fits(), "%s: %d workgroups are too many for one launch", what, groups);
    const bool eight = groups <= units + units / 16;
    const int waves = eight ? 8 : 4;
    const size_t lds = waves * 64 * sizeof(f32x4_t) + (size_t)M * (K + 8) * sizeof(bf16_t);
    bool refused = false;
    auto go = [&](auto kernel) {
        if (lds > 64 * 1024) refused = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess;
        if (!refused) hipLaunchKernelGGL(kernel, dim3(groups), dim3(waves * 64), lds, s, p.x, p.W, ln_w, ln_b, M, K, p.rows.packed(),
                                         Walk::packed(waves, 0, tail.d, TAIL && qkv_tail_plain_pairs(tail.rot, tail.d)), eps, p, tail);
    };
    auto by_rows = [&](auto ch) {
        constexpr int CH = decltype(ch)::value;
        if (eight && M <= 8) go(gemm_normed_kernel<8, CH, 1, TAIL>);
        else if (eight) go(gemm_normed_kernel<8, CH, 2, TAIL>);
        else if (M <= 8) go(gemm_normed_kernel<4, CH, 2, TAIL>);
        else go(gemm_normed_kernel<4, CH, 4, TAIL>);
    };
    switch ((K + 511) / 512) {
        case 1: by_rows(std::integral_constant<int, 1>{}); break;
        case 2: by_rows(std::integral_constant<int, 2>{}); break;
        case 3: by_rows(std::integral_constant<int, 3>{}); break;
        default: by_rows(std::integral_constant<int, 4>{}); break;
    }
    PTA_REQUIRE(!refused, "%s: %zu bytes of LDS were refused", what, lds);
    return pta_check_launch(what);
}

extern "C" int pta_gemm_normed_bf16(void* y, const void* x, const float* ln_w, const float* ln_b, float eps, const void* W,
                                    const float* bias, int M, int N, int K, int act, void* stream) {
    if (check_skinny("gemm_normed_bf16", y, x, W, M, N, K, act)) return 1;
    const SkinnyProblem p{y, (const bf16_t*)x, (const bf16_t*)W, bias, nullptr, nullptr, N, in_kernel(act) ? act : PTA_ACT_NONE, 0};
    if (launch_normed<false>("gemm_normed_bf16", p, ln_w, ln_b, eps, M, K, QkvTail{}, (hipStream_t)stream)) return 1;
    return in_kernel(act) ? 0 : pta_epilogue(y, N, nullptr, nullptr, nullptr, M, N, act, PTA_BF16, stream);
}

// The same with the tail of pta_gemm_skinny_qkv_bf16
extern "C" int pta_gemm_normed_qkv_bf16(void* q_out, const void* x, const float* ln_w, const float* ln_b, float eps, const void* W,
                                        const float* bias, const PtaRotation* rotation, const int* token_pos, const int* token_seq,
                                        const int* block_table, int bt_stride, void* k_pool, void* v_pool, int nh, int nkv, int d,
                                        int layout, int write_cache, int M, int K, void* stream) {
    SkinnyProblem p;
    QkvTail tail;
    if (make_tail_problem("gemm_normed_qkv_bf16", q_out, x, W, bias, rotation, token_pos, token_seq, block_table, bt_stride, k_pool,
                          v_pool, nh, nkv, d, layout, write_cache, M, K, p, tail)) return 1;
    return launch_normed<true>("gemm_normed_qkv_bf16", p, ln_w, ln_b, eps, M, K, tail, (hipStream_t)stream);
}

extern "C" int pta_gemm_skinny_glu_bf16(void* y, const void* x, const void* W, int M, int F, int K, int kind, float alpha, float limit,
                                        void* stream) {
    if (check_skinny("gemm_skinny_glu_bf16", y, x, W, M, F, K, PTA_ACT_NONE)) return 1;
    PTA_REQUIRE(M <= 16, "gemm_skinny_glu_bf16: at most 16 rows, got %d", M);
    PTA_REQUIRE(F < (1 << 30), "gemm_skinny_glu_bf16: %d features are too many", F);
    PTA_REQUIRE(kind == PTA_GLU_SILU || kind == PTA_GLU_CLAMPED || kind == PTA_GLU_GELU_TANH, "gemm_skinny_glu_bf16: kind %d is not built", kind);
    const int S = 2 * F >= 16384 ? pick_split(2 * F, K) : 2 * F >= 4096 ? 2 : 2 * F >= 1024 ? 4 : 8, units = pta_compute_units();
    int blocks = (F + 15) / 16;
    if (blocks > units) blocks = (blocks + units - 1) / units * units;  // a whole number of workgroups per unit (launch_cfg)
    static const int rot_env = getenv("PTA_SKINNY_ROT") ? atoi(getenv("PTA_SKINNY_ROT")) : -1;
    const int rot_stride = rot_env >= 0 ? rot_env : (K % 2048 == 0 ? 5 : 0);
    const Share rows(F, blocks);
    PTA_REQUIRE(rows.fits(), "gemm_skinny_glu_bf16: %d workgroups are too many for one launch", blocks);
    auto go = [&](auto kernel, size_t ring) {
        return launch_rings(kernel, dim3(blocks), dim3(S * 64), S * ring, (hipStream_t)stream, (const bf16_t*)x, (const bf16_t*)W, M, F, K, rows.packed(),
                            Walk::packed(S, rot_stride), (bf16_t*)y, kind, alpha, limit);
    };
    if (K > STREAM_MOST_K ? go(gemm_skinny_glu_kernel<0>, 2048)
                          : S <= 4 ? go(gemm_skinny_glu_kernel<4>, RowStream<2, 4>::RING) : go(gemm_skinny_glu_kernel<3>, RowStream<2, 3>::RING)) return 1;
    return pta_check_launch("gemm_skinny_glu_bf16");
}

// Two products of one launch: y1 = act1(x1 . W1^T + bias1), y2 = act2(x2 . W2^T + bias2), both [M, *] in
// bfloat16 with one K.  The waves per workgroup follow N1 + N2, so a product's bits differ from those of
// its own launch, but not with M or with what else is in the batch.
extern "C" int pta_gemm_skinny_pair_bf16(void* y1, const void* x1, const void* W1, const float* bias1, int N1, int act1,
                                         void* y2, const void* x2, const void* W2, const float* bias2, int N2, int act2,
                                         int M, int K, void* stream) {
    if (check_skinny("gemm_skinny_pair_bf16", y1, x1, W1, M, N1, K, act1)) return 1;
    if (check_skinny("gemm_skinny_pair_bf16", y2, x2, W2, M, N2, K, act2)) return 1;
    const SkinnyProblem a{y1, (const bf16_t*)x1, (const bf16_t*)W1, bias1, nullptr, nullptr, N1, in_kernel(act1) ? act1 : 0, 0};
    const SkinnyProblem b{y2, (const bf16_t*)x2, (const bf16_t*)W2, bias2, nullptr, nullptr, N2, in_kernel(act2) ? act2 : 0, 0};
    if (launch_skinny<bf16_t>(a, b, M, K, 0, 0, (hipStream_t)stream)) return 1;
    if (!in_kernel(act1) && pta_epilogue(y1, N1, nullptr, nullptr, nullptr, M, N1, act1, PTA_BF16, stream)) return 1;
    if (!in_kernel(act2) && pta_epilogue(y2, N2, nullptr, nullptr, nullptr, M, N2, act2, PTA_BF16, stream)) return 1;
    return 0;
}
