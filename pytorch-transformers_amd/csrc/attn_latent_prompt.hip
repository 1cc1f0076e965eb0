// Attention of prompts over a cache of latents, rows of 576 elements whose first 512 are the value (bfloat16 rows, 32-bit
// softmax and accumulation); what is computed is said in attn_latent.hip, other sizes and decode steps are attn_latent_mfma.h's.
//
// As there, a sequence's (new token, head) pairs are columns and all of them read the same rows.  A workgroup of four waves owns
// 64 columns, two pairs of waves 32 each, and walks the keys a page of 64 at a time:
//
//   S^T[64 keys x 32 cols] = K[64 x 576] . Q^T[576 x 32]         (32 keys a wave; A = cache rows, 36 steps of 16 elements)
//   online softmax over keys per column (32-bit; two lanes of each wave hold a column)
//   O^T[512 x 32 cols]    += V^T[512 x 64 keys] . P^T[64 x 32]   (256 elements a wave; A = the same rows, read transposed)
//
// The waves of a pair exchange a column's largest score and the weights through LDS, so that nothing is computed twice.  What
// bounds it is how often rows cross from LDS to the matrix cores, 68 KB for 68 products of 32 x 32 x 16: tiles of 32 columns
// halve that against sixteen.  A wave's queries (144 registers) and sums (128) then leave room for one wave a SIMD.  A page of
// rows is contiguous and goes straight to LDS, one page ahead, as it lies but for the order of the sixteen-byte pieces within
// each 128: piece p of row r lies at place p ^ turn(r), turn = bits 1, 2, 3 of r in reverse, so that both kinds of read spread
// over all banks: sixteen bytes of 32 rows at one place, and for V^T, by the transposing read (ds_read_tr16: sixteen lanes give the
// addresses of four rows of sixteen elements and get an element of the four rows each), 32 neighbours of four rows.  The order
// of keys within a step of 16 of the second product is the one in which the score tile's lanes hold them.
// A latent that is infinite or undefined changes no bit of a token that does not see it.
//
// Measured, launches in a row: two sequences of 1,500 and 1,900 tokens, 16 heads (102 GFLOP) 210 us, 490 TFLOP/s, where
// attn_latent_mfma.h's kernel takes 585; within the request, between other kernels, 231 us.  One of 2,048 132 / 427, eight of 64 to 700
// tokens 98 / 235 (there a workgroup's start, its queries above all, takes as long as its keys), one of 100 22 / 38.  Error against
// 64 bits: that kernel's to five digits.
#include "common.h"
#include "pta_kernels.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

#define LP_D 576            // elements of a row
#define LP_R 512            // of its value
#define LP_KEYS 64          // keys of a block: a page
#define LP_COLS 64          // columns of a workgroup
#define LP_STAGES 2
#define LP_ROW (LP_D * 2)               // bytes of a row
#define LP_STAGE (LP_KEYS * LP_ROW)     // 73,728: eighteen loads of sixteen bytes a thread
#define LP_LOADS (LP_STAGE / (256 * 16))
#define LP_WEIGHTS (LP_STAGES * LP_STAGE)    // after the stages: the waves' weights, 2 KB each
#define LP_MAXIMA (LP_WEIGHTS + 4 * 2048)    // and their columns' largest scores
#define LP_FLAGS (LP_MAXIMA + 4 * 32 * 4)    // and whether a wave found a value that is infinite or undefined
#define LP_LDS (LP_FLAGS + 4 * 4)
#define LP_LOG2E 1.4426950408889634f

struct LatentPromptArgs {
    void* out;  // [M, H, 512]
    const float* q;  // [M, H, 576]
    const bf16_t* k_pool;
    const int* block_table;
    int bt_stride;
    const int* cu_tokens;
    const int* seq_start;
    int H;
    float scale;
};

union LpFrag {
    uint4 u;
    bf16x8_t v;
    i16x4_t half[2];
};

__device__ __forceinline__ uint32_t lp_pack(float lo, float hi) {
    union { bf16x2_t b; uint32_t u; } c;
    c.b = __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t);
    return c.u;
}

// two neighbours of bfloat16, one of them infinite or undefined
__device__ __forceinline__ bool lp_special(uint32_t u) { return (u & 0x7f80u) == 0x7f80u || (u & 0x7f800000u) == 0x7f800000u; }

template <int N> __device__ __forceinline__ void lp_wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// sixteen bytes a lane straight to LDS, one lane after the other from `to` on; zeros past the buffer's end (no register is
// written; the waits are lp_wait_loads)
__device__ __forceinline__ void lp_fetch16(i32x4_t buffer, unsigned to, int at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(at), "s"(buffer) : "memory");
}

// a barrier behind the wave's own reads and writes of LDS; loads stay on their way
__device__ __forceinline__ void lp_meet() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <typename OutT>
__global__ __launch_bounds__(256, 1) void attn_latent_prompt_kernel(const LatentPromptArgs a) {
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    constexpr int KS = LP_D / 16, VT = LP_R / 64;  // steps of a row; value tiles of a wave
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pair = wave >> 1, kw = wave & 1;  // which columns; which half of the keys, and of the value
    const int c = lane & 31, h = lane >> 5;
    const int s = blockIdx.z, H = a.H;
    const int t0 = a.cu_tokens[s], n_new = a.cu_tokens[s + 1] - t0, start = a.seq_start[s];
    const int columns = n_new * H, groups = (columns + LP_COLS - 1) / LP_COLS;
    if ((int)blockIdx.x >= groups) return;
    const int row0 = (groups - 1 - (int)blockIdx.x) * LP_COLS;  // late tokens see the most keys: the longest work first
    const int wrow0 = row0 + pair * 32, rr = wrow0 + c;
    const bool valid = rr < columns;
    const int tq = valid ? rr / H : 0, head = valid ? rr - tq * H : 0;
    const int pos_q = valid ? start + tq : -1;  // -1: sees no key
    const long at_row = (long)(t0 + tq) * H + head;
    // (quotients come out of vector registers, of which there are none to spare)
    auto scalar = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const int k_end = scalar(start + min(n_new - 1, (row0 + LP_COLS - 1) / H) + 1);  // keys this workgroup walks
    const int all_see = scalar(wrow0 + 31 < columns ? start + wrow0 / H : -1);       // positions up to here every column sees
    const int first_pos = scalar(start + row0 / H);                                  // and every one of the workgroup that is a token's

    // staging: place p of a stage (sixteen bytes) is piece (p % 72, turned within its eight) of row p / 72; 32 rows on the same again
    auto turn = [](int r) { return ((r >> 1 & 1) << 2) | ((r >> 2 & 1) << 1) | (r >> 3 & 1); };
    int src[LP_LOADS / 2];
#pragma unroll
    for (int i = 0; i < LP_LOADS / 2; ++i) {
        const int p = i * 256 + tid, r = p / (LP_D / 8), piece = p - r * (LP_D / 8);
        src[i] = r * LP_ROW + (piece ^ turn(r)) * 16;
    }
    const int* bt = a.block_table + (long)s * a.bt_stride;
    const int blocks = (k_end + LP_KEYS - 1) / LP_KEYS;
    const unsigned to = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * 1024;
    auto fetch = [&](int b, int stage) {  // page b of the sequence; zeros past the last key
        const uint64_t at = (uint64_t)(uintptr_t)(a.k_pool + (long)bt[b] * (LP_KEYS * LP_D));
        const i32x4_t buffer{__builtin_amdgcn_readfirstlane((int)(uint32_t)at), __builtin_amdgcn_readfirstlane((int)((uint32_t)(at >> 32) & 0xffffu)),
                             __builtin_amdgcn_readfirstlane(min(LP_KEYS, k_end - b * LP_KEYS) * LP_ROW), 0x00020000};
#pragma unroll
        for (int i = 0; i < LP_LOADS; ++i)
            lp_fetch16(buffer, to + stage * LP_STAGE + i * 4096, src[i % (LP_LOADS / 2)] + i / (LP_LOADS / 2) * 32 * LP_ROW);
    };

    fetch(0, 0);

    // the pair's queries, scaled: column c, elements 16 step + 8 h .. + 7
    LpFrag qf[KS];
#pragma unroll
    for (int i = 0; i < KS; ++i) {
        float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
        if (valid) {
            lo = *reinterpret_cast<const float4*>(a.q + at_row * LP_D + i * 16 + h * 8);
            hi = *reinterpret_cast<const float4*>(a.q + at_row * LP_D + i * 16 + h * 8 + 4);
        }
        qf[i].u = make_uint4(lp_pack(lo.x * a.scale, lo.y * a.scale), lp_pack(lo.z * a.scale, lo.w * a.scale),
                             lp_pack(hi.x * a.scale, hi.y * a.scale), lp_pack(hi.z * a.scale, hi.w * a.scale));
    }

    // reads: K at step i, byte (i / 4) * 128 + the turned piece of eight; V^T tile t, half u of four keys likewise
    int k_at[4], v_at[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) k_at[i] = (32 * kw + c) * LP_ROW + (((2 * i) | h) ^ turn(c)) * 16;
    const int i16 = lane & 15, g16 = lane >> 4 & 1;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const int r = 8 * u + 4 * h + (i16 >> 2);  // (16 more a step: the same turn)
            v_at[u][o] = kw * LP_R + r * LP_ROW + ((4 * o + 2 * g16 + ((i16 & 3) >> 1)) ^ turn(r)) * 16 + (i16 & 1) * 8;
        }
    char* weights = lds + LP_WEIGHTS + pair * 4096 + lane * 16;            // [half of the keys][step][lane]
    float* maxima = (float*)(lds + LP_MAXIMA) + pair * 64 + c;             // [half of the keys][column]
    int* flags = (int*)(lds + LP_FLAGS);

    f32x16_t oacc[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[t][e] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    lp_wait_loads<0>();  // the first page
    lp_meet();
    for (int b = 0; b < blocks; ++b) {
        const int kb = b * LP_KEYS + 32 * kw;
        char* base = lds + (b & 1) * LP_STAGE;
        if (b + 1 < blocks) fetch(b + 1, (b + 1) & 1);
        f32x16_t sc;
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[e] = 0.f;
        LpFrag kf[2][4];
        auto read_k = [&](LpFrag (&dst)[4], int i0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[i].u = *reinterpret_cast<const uint4*>(base + k_at[i] + (i0 >> 2) * 128);
        };
        read_k(kf[0], 0);
#pragma unroll
        for (int i0 = 0; i0 < KS; i0 += 4) {
            if (i0 + 4 < KS) read_k(kf[((i0 >> 2) + 1) & 1], i0 + 4);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; ++i) sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[(i0 >> 2) & 1][i].v, qf[i0 + i].v, sc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the lane holds column c, keys kb + 8 (e / 4) + 4 h + e % 4
        if (kb + 31 > all_see) {
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (kb + 8 * (e >> 2) + 4 * h + (e & 3) > pos_q) sc[e] = -INFINITY;
        }
        float mx = sc[0];
#pragma unroll
        for (int e = 1; e < 16; ++e) mx = fmaxf(mx, sc[e]);
        mx = fold_32(mx, LaneMax());
        if (h == 0) maxima[kw * 32] = mx;
        // Rows r0 .. r1 - 1 are seen by some columns of the workgroup only (a few of its last page).  A value among them that is
        // infinite or undefined must reach those alone, and a weight of zero would not keep it from the others.
        const int r0 = max(first_pos + 1 - b * LP_KEYS, 0), r1 = min(k_end - b * LP_KEYS, LP_KEYS);
        if (r0 < r1) {
            bool found = false;
            for (int r = r0 + 2 * pair + h; r < r1; r += 4) {
                const uint4 u = *reinterpret_cast<const uint4*>(base + r * LP_ROW + kw * LP_R + c * 16);
                found |= lp_special(u.x) || lp_special(u.y) || lp_special(u.z) || lp_special(u.w);
            }
            found = __any(found);
            if (lane == 0) flags[wave] = found;
        }
        lp_meet();
        bool special = false;
        if (r0 < r1) special = __builtin_amdgcn_readfirstlane(flags[0] | flags[1] | flags[2] | flags[3]);
        // The first 32 keys count from the largest score up to them, the other 32 from the largest of all: a block's largest weight
        // is then exactly one in each half (with one reference for the 64, or one that lags behind, fewer weights are, and the
        // result's error against 64 bits grows by 0.5 and by 4 %).  Both waves of the pair see the same numbers.
        const float other = maxima[(kw ^ 1) * 32];
        const float mx0 = kw == 0 ? mx : other, mx1 = kw == 0 ? other : mx;
        const float m0 = fmaxf(m_run, mx0), m1 = fmaxf(m0, mx1);
        if (__any(mx0 > m_run)) {
            const float corr = __builtin_amdgcn_exp2f((m_run - (m0 == -INFINITY ? 0.f : m0)) * LP_LOG2E);
            l_run *= corr;
#pragma unroll
            for (int t = 0; t < VT; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) oacc[t][e] *= corr;
        }
        const bool raised = __any(mx1 > m0);
        const float corr1 = __builtin_amdgcn_exp2f((m0 - (m1 == -INFINITY ? 0.f : m1)) * LP_LOG2E);
        const float corr_l = m0 == -INFINITY ? 1.0f : corr1;  // (nothing is summed yet where no key has been seen)
        if (kw == 1) l_run *= corr_l;
        m_run = m1;
        const float m_mine = kw == 0 ? m0 : m1;
        const float m_use = m_mine == -INFINITY ? 0.f : m_mine * LP_LOG2E;
        LpFrag pf[2][2];
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2) {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[8 * k2 + 2 * e], LP_LOG2E, -m_use));
                const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[8 * k2 + 2 * e + 1], LP_LOG2E, -m_use));
                w[e] = lp_pack(p0, p1);
                l_run += __uint_as_float(w[e] << 16) + __uint_as_float(w[e] & 0xffff0000u);  // the weights as they were rounded
            }
            pf[0][k2].u = make_uint4(w[0], w[1], w[2], w[3]);
            *reinterpret_cast<uint4*>(weights + kw * 2048 + k2 * 1024) = pf[0][k2].u;
        }
        if (kw == 0) l_run *= corr_l;
        if (special) {  // (rare) such values are added where they are seen, by hand, and then stand as zeros for the products
            lp_meet();  // everyone's weights are there
            for (int r = r0; r < r1; ++r) {
                const bf16_t wb = *reinterpret_cast<const bf16_t*>(lds + LP_WEIGHTS + pair * 4096 + (r >> 5) * 2048 + (r >> 4 & 1) * 1024 +
                                                                   (c + 32 * (r >> 2 & 1)) * 16 + ((r >> 3 & 1) * 4 + (r & 3)) * 2);
                if (b * LP_KEYS + r > pos_q) continue;
                const float w = bf16_bits_to_f32(wb);
#pragma unroll
                for (int t = 0; t < VT; ++t)
#pragma unroll
                    for (int e = 0; e < 16; e += 4) {
                        const uint2 u = *reinterpret_cast<const uint2*>(base + r * LP_ROW + kw * LP_R + (t >> 1) * 128 +
                                                                        (((t & 1) * 4 + (e >> 2)) ^ turn(r)) * 16 + h * 8);
                        if (!(lp_special(u.x) || lp_special(u.y))) continue;
                        const uint32_t bits[4] = {u.x << 16, u.x & 0xffff0000u, u.y << 16, u.y & 0xffff0000u};
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if ((bits[i] & 0x7f800000u) == 0x7f800000u) oacc[t][e + i] += w * __uint_as_float(bits[i]);
                    }
            }
            lp_meet();
            for (int i = tid; i < (r1 - r0) * (LP_R / 4); i += 256) {
                uint2* at = reinterpret_cast<uint2*>(base + (r0 + i / (LP_R / 4)) * LP_ROW + i % (LP_R / 4) * 8);
                uint2 u = *at;
                if ((u.x & 0x7f80u) == 0x7f80u) u.x &= 0xffff0000u;
                if ((u.x & 0x7f800000u) == 0x7f800000u) u.x &= 0xffffu;
                if ((u.y & 0x7f80u) == 0x7f80u) u.y &= 0xffff0000u;
                if ((u.y & 0x7f800000u) == 0x7f800000u) u.y &= 0xffffu;
                *at = u;
            }
            lp_meet();
        }
        LpFrag vf[2][4];  // a tile's four steps of 16 keys
        auto read_v = [&](LpFrag (&dst)[4], int t) {
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4)
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    dst[k4].half[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(
                        base + v_at[u][t & 1] + k4 * 16 * LP_ROW + (t >> 1) * 128));
        };
        read_v(vf[0], 0);
        lp_meet();
#pragma unroll
        for (int k2 = 0; k2 < 2; ++k2) pf[1][k2].u = *reinterpret_cast<const uint4*>(weights + (kw ^ 1) * 2048 + k2 * 1024);
        if (kw == 1) {  // keys in their order
            const LpFrag x = pf[0][0], y = pf[0][1];
            pf[0][0] = pf[1][0], pf[0][1] = pf[1][1], pf[1][0] = x, pf[1][1] = y;
        }
#pragma unroll
        for (int t = 0; t < VT; ++t) {
            if (t + 1 < VT) read_v(vf[(t + 1) & 1], t + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k4 = 0; k4 < 4; ++k4) {
                if (k4 == 2 && raised) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) oacc[t][e] *= corr_l;
                }
                oacc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t & 1][k4].v, pf[k4 >> 1][k4 & 1].v, oacc[t], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        lp_wait_loads<0>();  // the next page has landed
        lp_meet();
    }
    float l = fold_32(l_run, LaneSum());
    if (h == 0) maxima[kw * 32] = l;
    lp_meet();
    l += maxima[(kw ^ 1) * 32];
    if (!valid) return;
    const float inv = 1.0f / l;
    OutT* to_row = (OutT*)a.out + at_row * LP_R + kw * (LP_R / 2) + 4 * h;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int e = 0; e < 16; e += 4) {  // elements 32 t + 8 (e / 4) + 4 h .. + 3 of the wave's half
            const float o[4] = {oacc[t][e] * inv, oacc[t][e + 1] * inv, oacc[t][e + 2] * inv, oacc[t][e + 3] * inv};
            if constexpr (sizeof(OutT) == 4) *reinterpret_cast<float4*>(to_row + t * 32 + e * 2) = make_float4(o[0], o[1], o[2], o[3]);
            else *reinterpret_cast<uint2*>(to_row + t * 32 + e * 2) = make_uint2(lp_pack(o[0], o[1]), lp_pack(o[2], o[3]));
        }
}

extern "C" int pta_attn_latent_prompt_ok(int R, int D) { return R == LP_R && D == LP_D ? 1 : 0; }

// out [M, H, 512] in 32-bit or bfloat16; steps in which sequences bring any number of tokens each (max_new at most)
extern "C" int pta_attn_latent_prompt(void* out, int out_bf16, const float* q, const void* k_pool, const int* block_table, int bt_stride,
                                      const int* cu_tokens, const int* seq_start, int n_seqs, int max_new, int M, int H, int R, int dr,
                                      float scale, void* stream) {
    PTA_REQUIRE(M > 0 && n_seqs > 0 && max_new > 0 && H > 0 && bt_stride > 0, "attn_latent_prompt: sizes must be positive");
    PTA_REQUIRE(out && q && k_pool && block_table && cu_tokens && seq_start, "attn_latent_prompt: null pointer");
    PTA_REQUIRE(pta_attn_latent_prompt_ok(R, R + dr), "attn_latent_prompt: rows of %d elements with %d of value are not built", R + dr, R);
    PTA_REQUIRE(n_seqs <= 65535 && (long)max_new * H < (1L << 31) - LP_COLS, "attn_latent_prompt: too many sequences or columns");
    for (const void* p : {(const void*)out, (const void*)q, k_pool})
        PTA_REQUIRE(((uintptr_t)p % 16) == 0, "attn_latent_prompt: pointers must be 16-byte aligned");
    const LatentPromptArgs a{out, q, (const bf16_t*)k_pool, block_table, bt_stride, cu_tokens, seq_start, H, scale};
    auto kern = out_bf16 ? attn_latent_prompt_kernel<bf16_t> : attn_latent_prompt_kernel<float>;
    constexpr int bytes = LP_LDS;
    static_assert(LP_LDS <= 160 * 1024 && LP_KEYS == PTA_PAGE, "two pages of rows must fit LDS");
    // (on every device: the attribute belongs to the device that is current)
    PTA_REQUIRE(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess,
                "attn_latent_prompt: %d bytes of LDS were refused", bytes);
    const dim3 grid((unsigned)(((long)max_new * H + LP_COLS - 1) / LP_COLS), 1, n_seqs);
    hipLaunchKernelGGL(kern, grid, dim3(256), bytes, (hipStream_t)stream, a);
    return pta_check_launch("attn_latent_prompt");
}
