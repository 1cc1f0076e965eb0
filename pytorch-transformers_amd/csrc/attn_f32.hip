// Causal attention over the paged cache in true 32-bit, on the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32: products
// and sums in 32-bit), for head sizes that are a multiple of 4.  What it computes is what attn_generic.hip says.
//
// Sixteen (token, head) pairs that share a KV head are the sixteen columns of a tile.  A page of 64 keys is one unit of work:
// scores = K . q^T (four tiles of sixteen keys), the columns' maxima, weights and their sums, and V^T . weights.  The scores'
// registers are the second product's operand as they are (a lane holds four keys of its column in both), so nothing goes
// through LDS on the way.  A page's result (maximum, sum, weighted values) is joined to what the pages before it gave, page
// by page in order, whoever computed them: what a token gets does not depend on the step's cut, on its batch or on the kernel.
//
// 71 heads of 64 on one KV head, four prompts of 90 to 700 tokens in a launch: 5,952 us with a wave per (token, head), 224 us.
//
// A tile's columns belong to one sequence (cu_tokens): a wave whose columns came from as many sequences walked their contexts
// one after the other (32 single tokens behind 1,000 keys beside a prompt of 64, 16 heads on 16 KV heads: 5,770 us, now 111; 135
// with a wave per token and head).
//   prompts: a wave owns one or two tiles and walks their pages.  Bound by the matrix instruction and by L2 (a page of heads
//     of 64 is 32 KB a tile); the tiles with the most keys start first.
//   single tokens, or a few behind many (pta_attn_f32_plan): the waves of a workgroup share the pages of a tile out and meet
//     in LDS.
#include "common.h"
#include "pta_kernels.h"
#include "score_bias.h"

#include <algorithm>

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct AttnF32 {
    float* out;
    const float* q;
    const float* k_pool;
    const float* v_pool;
    const int* block_table;
    int bt_stride;
    const int* token_seq;
    const int* token_pos;
    const float* slopes;
    int bias_mode;
    float bias_scale;
    int M, nh, nkv, d;
    float scale;
    int window, chunk;
    const float* sink;
    PtaHeadRows rows;
    int vec;  // heads may be written sixteen bytes at a time
    const int* cu_tokens;  // first token of every sequence of the step, and their number; or null: every token by itself
    int n_seqs;
    int share_new;         // sequences of up to so many new tokens go to the workgroups that share pages out
};

// a column: its token's keys first .. nkeys - 1 of sequence seq (nkeys 0: no such column)
struct Column {
    int token, head, seq, first, nkeys;
    float slope;
};

__device__ __forceinline__ Column column_of(const AttnF32& a, int token, int head, bool there) {
    Column c{0, 0, -1, 0, 0, 0.f};
    if (!there) return c;
    c.token = token, c.head = head, c.seq = a.token_seq[token], c.nkeys = a.token_pos[token] + 1;
    if (a.window > 0) c.first = max(0, c.nkeys - a.window);
    if (a.chunk > 0) c.first = max(c.first, (c.nkeys - 1) / a.chunk * a.chunk);
    if (a.slopes) c.slope = a.slopes[head];
    return c;
}

// query operands of a column: four elements from 16 b + kq on, zeros past the head
template <int DT>
__device__ __forceinline__ void load_query(const AttnF32& a, const Column& c, int kq, f32x4 (&q)[DT]) {
    const float* row = a.q + ((long)c.token * a.nh + c.head) * a.d;
#pragma unroll
    for (int b = 0; b < DT; ++b) {
        q[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (c.nkeys > 0 && 16 * b + kq < a.d) q[b] = *(const f32x4*)(row + 16 * b + kq);
    }
}

// One page for CT tiles: m, l and o of its keys alone.  ``seen[c]``: whether column c looks at this page's sequence at all.
// ``end``: keys of the sequence that any column of the wave sees (what lies behind is whatever the page held before).  ``spare``:
// LDS of the wave's own for the weights of the page.
template <int DT, int CT>
__device__ __forceinline__ void page_pass(const AttnF32& a, const float* kp, const float* vp, int j0, int end, const f32x4 (&q)[CT][DT],
                                          const Column (&col)[CT], const bool (&seen)[CT], float (&m)[CT], float (&l)[CT],
                                          f32x4 (&o)[CT][DT], float* spare) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = 4 * (lane >> 4);
    f32x4 s[CT][4];
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int t = 0; t < 4; ++t) s[c][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const float* row = kp + (16 * t + r16) * a.d + kq;
        f32x4 k[DT];
#pragma unroll
        for (int b = 0; b < DT; ++b) {
            k[b] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (16 * b + kq < a.d) k[b] = *(const f32x4*)(row + 16 * b);
        }
#pragma unroll
        for (int b = 0; b < DT; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < CT; ++c) s[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[b][e], q[c][b][e], s[c][t], 0, 0, 0);
    }
    bool whole = true;  // every column sees every key of the page
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int first = seen[c] ? col[c].first : 0, n = seen[c] ? col[c].nkeys : 0;
        whole = whole && first <= j0 && n >= j0 + PTA_PAGE;
        float top = -INFINITY;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = j0 + 16 * t + kq + e;
                float v = s[c][t][e] * a.scale;
                if (a.slopes)  // slope x key position as the reference rounds it (0), exact (1), or x the distance from the query (2)
                    v += (a.bias_mode == 0 ? round_to_bf16(col[c].slope * round_to_bf16((float)j))
                                           : col[c].slope * (float)(a.bias_mode == 2 ? j - (col[c].nkeys - 1) : j)) * a.bias_scale;
                v = j >= first && j < n ? v : -INFINITY;
                s[c][t][e] = v;
                top = fmaxf(top, v);
            }
        top = column_max(top);
        const float base = top == -INFINITY ? 0.f : top;
        float sum = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = j0 + 16 * t + kq + e;
                const float p = j >= first && j < n ? expf(s[c][t][e] - base) : 0.f;
                s[c][t][e] = p;
                sum += p;
            }
        m[c] = top, l[c] = column_sum(sum);
    }
    const bool ragged = __ballot(!whole) != 0;
#pragma unroll
    for (int b = 0; b < DT; ++b) {
        const int row = min(16 * b + r16, a.d - 1);  // rows past the head: read again, not kept
        f32x4 v[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = *(const f32x4*)(vp + row * PTA_PAGE + 16 * t + kq);
#pragma unroll
        for (int c = 0; c < CT; ++c) o[c][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        bool odd = false;
        if (ragged) {
            // A weight of 0 must hide its value whatever that is.  Keys behind the end are cleared; an infinite or undefined
            // value is cleared too and joins below those columns alone that see its key.
            float zero = 0.f;
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (j0 + 16 * t + kq + e >= end) v[t][e] = 0.f;
                    zero += v[t][e] * 0.f;
                }
            odd = __ballot(!(zero == 0.f)) != 0;
            if (odd) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (!(v[t][e] * 0.f == 0.f)) v[t][e] = 0.f;
            }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < CT; ++c) o[c][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][e], s[c][t][e], o[c][b], 0, 0, 0);
        if (odd) {  // (rare: the columns' weights go through LDS, so that this is a loop and little code)
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) spare[(c * PTA_PAGE + 16 * t + kq + e) * 16 + r16] = s[c][t][e];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 1
            for (int j = 0; j < PTA_PAGE; ++j) {
                float x[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = vp[min(16 * b + kq + i, a.d - 1) * PTA_PAGE + j];
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    if (!seen[c] || j0 + j < col[c].first || j0 + j >= col[c].nkeys) continue;
                    const float p = spare[(c * PTA_PAGE + j) * 16 + r16];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (!(x[i] * 0.f == 0.f)) o[c][b][i] += p * x[i];
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// what the pages so far gave (M, L, O) takes in one more page's result; a page with no key of the column changes nothing
__device__ __forceinline__ bool join(float& M, float& L, float m, float l, float& keep, float& take) {
    if (m == -INFINITY && l == 0.f) return false;
    const float top = fmaxf(M, m);
    keep = expf(M - top), take = expf(m - top);  // the first page: M is -infinity, keep 0
    L = L * keep + l * take;
    M = top;
    return true;
}

__device__ __forceinline__ void store_heads(const AttnF32& a, const Column& c, int dim, f32x4 v) {
    float* to = a.out + (long)c.token * a.rows.ld + (long)c.head * a.rows.head + dim;
    if (a.vec) {
        if (dim < a.rows.keep) *(f32x4*)to = v;
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (dim + i < a.rows.keep) to[i] = v[i];
    }
}

// a learned number per head: its exponential joins the sum of the weights once, with no key and no value
__device__ __forceinline__ float last_factor(const AttnF32& a, const Column& c, float M, float L) {
    float last = 1.f;
    if (a.sink) {
        const float top = fmaxf(M, a.sink[c.head]);
        last = expf(M - top);
        L = L * last + expf(a.sink[c.head] - top);
    }
    return last / L * a.rows.mult;
}

// the keys that a wave's columns see: from the first of any to the last of any
template <int CT>
__device__ __forceinline__ void keys_of(const Column (&col)[CT], int& from, int& end) {
    from = 0x7fffffff, end = 0;
#pragma unroll
    for (int c = 0; c < CT; ++c)
        if (col[c].nkeys > 0) from = min(from, col[c].first), end = max(end, col[c].nkeys);
#pragma unroll
    for (int x = 1; x < 16; x <<= 1) from = min(from, __shfl_xor(from, x)), end = max(end, __shfl_xor(end, x));
    from = __builtin_amdgcn_readfirstlane(from), end = __builtin_amdgcn_readfirstlane(end);
}

template <int DT, int CT>
__global__ __launch_bounds__(256, DT <= 6 ? 2 : 1) void attn_f32_prompt_kernel(AttnF32 a, int tiles) {
    __shared__ float weights[4][CT * PTA_PAGE * 16];
    float* spare = weights[threadIdx.x >> 6];
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = 4 * (lane >> 4);
    const int per = a.nh / a.nkv, kvh = blockIdx.y;
    // the last tiles of a sequence have the most keys and start first
    int tile = tiles - 1 - ((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6)), seq = 0, n_new = 0;
    if (tile < 0) return;
    for (;; seq += 64) {  // 64 sequences at a time: whose tile this is
        if (seq >= a.n_seqs) return;
        int n = 0, own = 0;
        if (seq + lane < a.n_seqs) {
            n = a.cu_tokens[seq + lane + 1] - a.cu_tokens[seq + lane];
            if (n > a.share_new) own = (int)(((long)n * per + 16 * CT - 1) / (16 * CT));
        }
        int upto = own;
#pragma unroll
        for (int x = 1; x < 64; x <<= 1) {
            const int before = __shfl_up(upto, x);
            if (lane >= x) upto += before;
        }
        const unsigned long long past = __ballot(upto > tile);
        if (past) {
            const int who = __ffsll(past) - 1;
            tile -= __shfl(upto - own, who);
            n_new = __shfl(n, who);
            seq += who;
            break;
        }
        tile -= __shfl(upto, 63);
    }
    seq = __builtin_amdgcn_readfirstlane(seq);
    const int t0 = a.cu_tokens[seq];
    Column col[CT];
    f32x4 q[CT][DT], O[CT][DT];
    float M[CT], L[CT];
    bool seen[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        // columns are (token, head of the group) pairs in a row
        const long at = ((long)tile * CT + c) * 16 + r16;
        col[c] = column_of(a, t0 + (int)(at / per), kvh * per + (int)(at % per), at < (long)n_new * per);
        seen[c] = col[c].nkeys > 0;
        load_query<DT>(a, col[c], kq, q[c]);
        M[c] = -INFINITY, L[c] = 0.f;
#pragma unroll
        for (int b = 0; b < DT; ++b) O[c][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    int from, end;
    keys_of(col, from, end);
    const int* bt = a.block_table + (long)seq * a.bt_stride;
    for (int p = from / PTA_PAGE; p * PTA_PAGE < end; ++p) {
        const long at = ((long)bt[p] * a.nkv + kvh) * PTA_PAGE * a.d;
        float m[CT], l[CT], keep, take;
        f32x4 o[CT][DT];
        page_pass<DT, CT>(a, a.k_pool + at, a.v_pool + at, p * PTA_PAGE, end, q, col, seen, m, l, o, spare);
#pragma unroll
        for (int c = 0; c < CT; ++c)
            if (join(M[c], L[c], m[c], l[c], keep, take)) {
#pragma unroll
                for (int b = 0; b < DT; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) O[c][b][i] = fmaf(O[c][b][i], keep, o[c][b][i] * take);
            }
    }
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        if (col[c].nkeys == 0) continue;
        const float f = last_factor(a, col[c], M[c], L[c]);
#pragma unroll
        for (int b = 0; b < DT; ++b) store_heads(a, col[c], 16 * b + kq, O[c][b] * f);
    }
}

template <int DT, int NW>
__global__ __launch_bounds__(NW * 64) void attn_f32_shared_kernel(AttnF32 a) {
    __shared__ f32x4 po[NW][DT][64];
    __shared__ float pm[NW][16], pl[NW][16];
    __shared__ float weights[NW][PTA_PAGE * 16];
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = 4 * (lane >> 4), wave = threadIdx.x >> 6;
    float* spare = weights[wave];
    const int per = a.nh / a.nkv, kvh = blockIdx.y, run = blockIdx.x;
    int t0 = run, n_new = 1;
    if (a.cu_tokens) {
        t0 = a.cu_tokens[run], n_new = a.cu_tokens[run + 1] - t0;
        if (n_new > a.share_new) return;
    }
    if ((long)blockIdx.z * 16 >= (long)n_new * per) return;
    const int at0 = blockIdx.z * 16 + r16;
    Column col[1] = {column_of(a, t0 + at0 / per, kvh * per + at0 % per, at0 < (long)n_new * per)};
    f32x4 q[1][DT], O[(DT + NW - 1) / NW];
    load_query<DT>(a, col[0], kq, q[0]);
    const bool seen[1] = {col[0].nkeys > 0};
    int from, end;
    keys_of(col, from, end);
    const int* bt = a.block_table + (long)__builtin_amdgcn_readfirstlane(col[0].seq) * a.bt_stride;  // (column 0 is always there)
    const int p0 = from / PTA_PAGE, p1 = (end + PTA_PAGE - 1) / PTA_PAGE;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int i = 0; i < (DT + NW - 1) / NW; ++i) O[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int p = p0; p < p1; p += NW) {
        const int n = min(NW, p1 - p);
        if (wave < n) {
            const long at = ((long)bt[p + wave] * a.nkv + kvh) * PTA_PAGE * a.d;
            float m[1], l[1];
            f32x4 o[1][DT];
            page_pass<DT, 1>(a, a.k_pool + at, a.v_pool + at, (p + wave) * PTA_PAGE, end, q, col, seen, m, l, o, spare);
#pragma unroll
            for (int b = 0; b < DT; ++b) po[wave][b][lane] = o[0][b];
            if (lane < 16) pm[wave][lane] = m[0], pl[wave][lane] = l[0];
        }
        __syncthreads();
        for (int w = 0; w < n; ++w) {  // in the pages' order; every wave the rows that it will write
            float keep, take;
            if (join(M, L, pm[w][r16], pl[w][r16], keep, take)) {
#pragma unroll
                for (int i = 0; i < (DT + NW - 1) / NW; ++i) {
                    const int b = wave + i * NW;
                    if (b < DT) {
                        const f32x4 o = po[w][b][lane];
#pragma unroll
                        for (int e = 0; e < 4; ++e) O[i][e] = fmaf(O[i][e], keep, o[e] * take);
                    }
                }
            }
        }
        __syncthreads();
    }
    if (col[0].nkeys == 0) return;
    const float f = last_factor(a, col[0], M, L);
#pragma unroll
    for (int i = 0; i < (DT + NW - 1) / NW; ++i) {
        const int b = wave + i * NW;
        if (b < DT) store_heads(a, col[0], 16 * b + kq, O[i] * f);
    }
}

template <int DT>
static void launch(const AttnF32& a, int shared_tiles, int prompt_waves, int wave_tiles, hipStream_t s) {
    constexpr int NW = DT <= 4 ? 8 : DT <= 8 ? 4 : 2;
    const int runs = a.cu_tokens ? a.n_seqs : a.M;
    // sequences side by side: most have fewer tiles than the largest, and the dies are given workgroups in turn (32 single
    // tokens of 1,000 keys beside one prompt of 16 tiles, tiles side by side: 570 us, all of them on one die)
    if (shared_tiles > 0)
        hipLaunchKernelGGL((attn_f32_shared_kernel<DT, NW>), dim3(runs, a.nkv, shared_tiles), dim3(NW * 64), 0, s, a);
    const dim3 grid((prompt_waves + 3) / 4, a.nkv);
    if (prompt_waves > 0 && wave_tiles == 1)
        hipLaunchKernelGGL((attn_f32_prompt_kernel<DT, 1>), grid, dim3(256), 0, s, a, prompt_waves);
    else if (prompt_waves > 0)
        hipLaunchKernelGGL((attn_f32_prompt_kernel<DT, DT <= 4 ? 2 : 1>), grid, dim3(256), 0, s, a, prompt_waves);
}

// How a step's sequences (new tokens and cached ones of each) are given to the two kernels.
extern "C" int pta_attn_f32_plan(const int* new_tokens, const int* starts, int n_seqs, int nh, int nkv, int d, PtaAttnF32Plan* plan) {
    PTA_REQUIRE(new_tokens && starts && plan && n_seqs > 0, "attn_f32_plan: no sequences or a null pointer");
    PTA_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0 && d > 0, "attn_f32_plan: sizes must be positive and heads a multiple of kv heads (nh=%d nkv=%d d=%d)", nh, nkv, d);
    const long per = nh / nkv;
    // sequences of up to `limit` new tokens: tiles of the largest, of all, and the most pages
    long most, all, pages;
    auto upto = [&](int limit) {
        most = all = pages = 0;
        for (int i = 0; i < n_seqs; ++i) {
            if (new_tokens[i] <= 0 || new_tokens[i] > limit) continue;
            const long tiles = (new_tokens[i] * per + 15) / 16;
            most = std::max(most, tiles), all += tiles;
            pages = std::max(pages, ((long)starts[i] + new_tokens[i] + PTA_PAGE - 1) / PTA_PAGE);
        }
    };
    // Sharing shortens a tile's chain of pages, but a workgroup that shares takes a compute unit (heads up to 64) or half of
    // one.  Shared / a wave a tile, us: 64 tokens of 16 heads of 64 on 16 KV heads, 4 rounds of such workgroups: 128 keys 44 / 30, 256
    // keys 56 / 43; 8 x 64 tokens behind 1,000 keys, 2 rounds: 69 / 106; 1,000 tokens, 4 rounds: 71 / 99; 64 x 16 tokens of 32 heads
    // of 128 on 8 behind 128 keys, 4 rounds: 91 / 74; 8 x 256 tokens of it behind 256 keys, 8 rounds: 286 / 322, behind 4,000 keys:
    // 2,238 / 2,932; 8 x 64 tokens of 71 heads of 64 on one behind 128 keys, 9 rounds: 91 / 50.
    const long fit = d <= 64 ? 256 : 512, waves_each = d <= 64 ? 8 : 4;
    const int limits[] = {0x7fffffff, 256, 64, 16, 4, 1, 0};
    for (int limit : limits) {
        plan->share_new = limit;
        upto(limit);
        if (4 * all * nkv <= fit * (pages < 2 * waves_each ? 5 : d <= 64 ? 20 : 256)) break;
    }
    plan->shared_tiles = (int)most;
    long waves[2] = {0, 0};
    for (int i = 0; i < n_seqs; ++i)
        for (int t = 0; t < 2; ++t)
            if (new_tokens[i] > plan->share_new) waves[t] += (new_tokens[i] * per + 16 * (t + 1) - 1) / (16 * (t + 1));
    // two tiles a wave read a page once for both; one has the shorter chain and leaves no columns empty in short runs: 8 x 256
    // tokens of 71 heads on one KV head, 9,088 tiles: 116 us with two, 128 with one; 1,000 tokens of 16 on 16, 1,008: 142 and 99
    plan->wave_tiles = d > 64 || 5 * waves[1] > 3 * waves[0] || waves[0] * nkv < 4096 ? 1 : 2;
    PTA_REQUIRE(waves[plan->wave_tiles - 1] <= 0x7fffffff - 3, "attn_f32_plan: too many tokens for one launch");
    plan->prompt_waves = (int)waves[plan->wave_tiles - 1];
    return 0;
}

// cu_tokens null: every token by itself; else plan is pta_attn_f32_plan's for these sequences
extern "C" int pta_attn_f32(float* out, const float* q, const float* k_pool, const float* v_pool, const int* block_table,
                            int bt_stride, const int* token_seq, const int* token_pos, const PtaScoreBias* score_bias, int M,
                            int nh, int nkv, int d, float scale, int window, int chunk, const float* sink,
                            const PtaHeadRows* head_rows, const int* cu_tokens, int n_seqs, const PtaAttnF32Plan* plan,
                            void* stream) {
    int bias_mode = 0;
    if (pta_score_bias_mode("attn_f32", score_bias, &bias_mode)) return 1;
    const float* slopes = score_bias ? score_bias->slopes : nullptr;
    PTA_REQUIRE(M > 0 && nh > 0 && nkv > 0 && nh % nkv == 0, "attn_f32: sizes must be positive and heads a multiple of kv heads (M=%d nh=%d nkv=%d)",
                M, nh, nkv);
    PTA_REQUIRE(d > 0 && d <= 256 && d % 4 == 0, "attn_f32: head size %d is no multiple of 4 up to 256", d);
    PTA_REQUIRE(nkv <= 65535 && nh / nkv <= 65535 * 16, "attn_f32: %d heads on %d kv heads are too many", nh, nkv);
    PTA_REQUIRE(!cu_tokens || (plan && n_seqs > 0 && plan->shared_tiles >= 0 && plan->shared_tiles <= 65535 && plan->prompt_waves >= 0 && (plan->wave_tiles == 1 || (plan->wave_tiles == 2 && d <= 64))),
                "attn_f32: %d sequences without a plan for them", n_seqs);
    PTA_REQUIRE(window >= 0 && chunk >= 0, "attn_f32: window and chunk must be 0 (none) or positive, got %d and %d", window, chunk);
    PTA_REQUIRE((uintptr_t)q % 16 == 0 && (uintptr_t)k_pool % 16 == 0 && (uintptr_t)v_pool % 16 == 0,
                "attn_f32: queries and pages must be sixteen-byte aligned");
    const PtaHeadRows rows = pta_head_rows_of(head_rows, nh, d);
    if (pta_check_head_rows("attn_f32", rows, nh, d, out, 1)) return 1;
    const int vec = rows.keep % 4 == 0 && rows.head % 4 == 0 && rows.ld % 4 == 0 && (uintptr_t)out % 16 == 0;
    const AttnF32 a{out, q, k_pool, v_pool, block_table, bt_stride, token_seq, token_pos, slopes, bias_mode,
                    slopes ? score_bias->scale : 0.f, M, nh, nkv, d, scale, window, chunk, sink, rows, vec, cu_tokens, n_seqs, cu_tokens ? plan->share_new : 1};
    hipStream_t s = (hipStream_t)stream;
    const int dt = (d + 15) / 16;
    const int shared = cu_tokens ? plan->shared_tiles : (nh / nkv + 15) / 16, waves = cu_tokens ? plan->prompt_waves : 0;
    const int wave_tiles = cu_tokens ? plan->wave_tiles : 1;
    if (dt <= 1) launch<1>(a, shared, waves, wave_tiles, s);
    else if (dt <= 2) launch<2>(a, shared, waves, wave_tiles, s);
    else if (dt <= 3) launch<3>(a, shared, waves, wave_tiles, s);
    else if (dt <= 4) launch<4>(a, shared, waves, wave_tiles, s);
    else if (dt <= 5) launch<5>(a, shared, waves, wave_tiles, s);
    else if (dt <= 6) launch<6>(a, shared, waves, wave_tiles, s);
    else if (dt <= 8) launch<8>(a, shared, waves, wave_tiles, s);
    else launch<16>(a, shared, waves, wave_tiles, s);
    return pta_check_launch("attn_f32");
}
