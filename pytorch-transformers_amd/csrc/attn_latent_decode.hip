// Decode steps of attention over a cache of latents (attn_latent.hip says what is computed): bfloat16 cache rows of D = R + dr
// elements, one new token per sequence, in three launches instead of eight.
//
//   latent_queries   each head's plain query through its key expansion into the first R of its frame, the rotated parts and the
//                    token's cache row (what latent_prep does) by further workgroups of the same launch
//   latent_pages     a workgroup per (sequence, range of keys, sixteen heads): a page of 64 rows is staged in LDS as it lies and
//                    serves scores and values; leaves unnormed sums per range
//   latent_values    merges a token's ranges and takes the result through the head's value expansion
//
// What bounds a layer here is launches and chains of dependent loads, not bytes: 16 heads, R = 512, dr = 64, 8 sequences of 64 to
// 700 keys took 72 us a layer in eight launches (two of them the vendor library's, three copies), and takes 20 in three (4.6,
// 9.2 and 5.8).
#include "attn_latent_token.h"

typedef __bf16 ld_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ld_f32x4 __attribute__((ext_vector_type(4)));
typedef short ld_i16x4 __attribute__((ext_vector_type(4)));

union LdFrag {
    uint4 u;
    ld_bf16x8 v;
    ld_i16x4 half[2];
};

// ---- queries ------------------------------------------------------------------------------------------------------------
// Workgroups below `expand`: 64 rows of one head's turned key expansion kt [H][R][dn], sixteen a wave, held in registers (KC
// pieces of 32 elements), for every sixteen tokens in turn.  Behind them a workgroup a token for its rotated parts, then one a
// token for its cache row.
template <int KC>
__global__ __launch_bounds__(256) void latent_queries_kernel(float* __restrict__ q_full, bf16_t* __restrict__ k_pool,
                                                             const bf16_t* __restrict__ q_rows, long q_ld,
                                                             const bf16_t* __restrict__ kt, LatentToken t, int M, int expand) {
    __shared__ float red[16];
    if ((int)blockIdx.x >= expand) {
        const int m = (int)blockIdx.x - expand;
        if (m < M) latent_rotations<bf16_t>(t, m, q_full, q_rows, q_ld);
        else latent_row<bf16_t>(t, m - M, k_pool, red);
        return;
    }
    const int D = t.R + t.dr, lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const int per = (t.R + 63) / 64, h = blockIdx.x / per, r0 = (blockIdx.x % per) * 64 + (threadIdx.x >> 6) * 16;
    if (r0 >= t.R) return;
    LdFrag w[KC];
    const bf16_t* row = kt + ((long)h * t.R + min(r0 + r16, t.R - 1)) * t.dn + g * 8;
#pragma unroll
    for (int c = 0; c < KC; ++c) w[c].u = *(const uint4*)(row + 32 * c);
    for (int m0 = 0; m0 < M; m0 += 16) {
        const int m = m0 + r16;
        const bf16_t* qr = q_rows + (long)min(m, M - 1) * q_ld + (long)h * (t.dn + t.dr) + g * 8;
        LdFrag q[KC];
#pragma unroll
        for (int c = 0; c < KC; ++c) q[c].u = *(const uint4*)(qr + 32 * c);
        ld_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; ++c) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c].v, q[c].v, acc, 0, 0, 0);
        // element i: row r0 + 4 g + i of the expansion, token m
        if (m < M && r0 + 4 * g < t.R) *(ld_f32x4*)(q_full + ((long)m * t.H + h) * D + r0 + 4 * g) = acc;
    }
}

// ---- pages --------------------------------------------------------------------------------------------------------------
#define LP_PIECES 20  // D <= 640
#define LP_QUERIES 5  // pieces of sixteen queries a thread takes: 16 D / 8 / 256

// TILES: sixteen-element tiles of the value part a wave holds (its quarter of them)
template <int TILES>
__global__ __launch_bounds__(256) void latent_pages_kernel(
    // what a workgroup's loads are found by: the first fourteen words, which are in registers when it starts
    const float* __restrict__ queries,  // [M, H, D]
    const bf16_t* __restrict__ k_pool, const int* __restrict__ block_table, const int* __restrict__ seq_start, int bt_stride, int size, int splits, int H, int D,
    int R,  // size: keys a range (whole pages); splits: ranges
    float scale,
    float* __restrict__ po,    // [M, H, splits, R] sums of weights times rows, not normed
    float* __restrict__ pm,    // [M, H, splits] maxima
    float* __restrict__ pl) {  // [M, H, splits] sums of weights
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    const int P = D + 8;               // row distance in LDS: neighbouring rows start in other banks
    bf16_t* Ks = lds;                  // [64][P]
    bf16_t* Qs = Ks + 64 * P;          // [16][P]
    bf16_t* Ps = Qs + 16 * P;          // [16 columns][72] weights of the page's keys
    float* stat = (float*)(Ps + 16 * 72);  // [4][16] maxima, [4][16] sums
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int s = blockIdx.z, split = blockIdx.y, h0 = blockIdx.x * 16;
    const int k0 = split * size;
    // the range's first page beside the sequence's length, not behind it (an entry past the sequence's pages is read but not used)
    const int* bt = block_table + (long)s * bt_stride;
    int first_page = bt[min(k0 / PTA_PAGE, bt_stride - 1)], nkeys = seq_start[s] + 1;
    asm volatile("" : "+s"(first_page), "+s"(nkeys));
    const int k1 = min(nkeys, k0 + size);
    const long row = (long)s * H + h0 + r16;  // this lane's column (a head past H: read as the last one, not kept)
    const bool there = h0 + r16 < H;
    ld_f32x4 acc[TILES];
#pragma unroll
    for (int i = 0; i < TILES; ++i) acc[i] = ld_f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    if (k0 < k1) {
        const int pieces = D / 8, per = pieces / 4;  // sixteen-byte pieces of a row (D is a multiple of 32), of a page per thread
        // Piece tid + 256 j of a page's 64 rows, which are one run of memory, lies in row (tid + 256 j) / pieces: the row and the
        // piece in it are moved on instead of divided for.  All of a page's loads are in flight together, the next page's
        // behind this one's arithmetic.
        const int step_row = 256 / pieces, step_at = 256 % pieces, row0 = tid / pieces, at0 = tid % pieces;
        uint4 pre[LP_PIECES];
        auto fetch = [&](int kb) {
            const uint4* page = (const uint4*)(k_pool + (long)(kb == k0 ? first_page : bt[kb / PTA_PAGE]) * PTA_PAGE * D) + tid;
#pragma unroll
            for (int j = 0; j < LP_PIECES; ++j)
                if (j < per) pre[j] = page[256 * j];
        };
        // Queries, scaled and rounded, once for the four waves: all asked for before the page and in LDS while it comes (a piece after the other behind
        // the page: 1.1 us more, 16 heads, R = 512, 8 sequences of 64 to 700 keys)
        float4 lo[LP_QUERIES], hi[LP_QUERIES];
        {
            int c = row0, e = at0;
#pragma unroll
            for (int j = 0; j < LP_QUERIES; ++j) {
                const float* src = queries + ((long)s * H + min(h0 + min(c, 15), H - 1)) * D + 8 * e;
                lo[j] = *(const float4*)src, hi[j] = *(const float4*)(src + 4);
                c += step_row, e += step_at;
                if (e >= pieces) e -= pieces, ++c;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch(k0);
        __builtin_amdgcn_sched_barrier(0);
        {
            int c = row0, e = at0;
#pragma unroll
            for (int j = 0; j < LP_QUERIES; ++j) {
                const float v[8] = {lo[j].x * scale, lo[j].y * scale, lo[j].z * scale, lo[j].w * scale,
                                    hi[j].x * scale, hi[j].y * scale, hi[j].z * scale, hi[j].w * scale};
                if (tid + 256 * j < 16 * pieces) *(uint4*)(Qs + c * P + 8 * e) = pack8(v);
                c += step_row, e += step_at;
                if (e >= pieces) e -= pieces, ++c;
            }
        }
        for (int kb = k0; kb < k1; kb += PTA_PAGE) {
            if (kb > k0) __syncthreads();  // the last page's reads are done
            {   // what lies behind the sequence's end is cleared
                int k = row0, e = at0;
#pragma unroll
                for (int j = 0; j < LP_PIECES; ++j)
                    if (j < per) {
                        *(uint4*)(Ks + k * P + 8 * e) = kb + k < k1 ? pre[j] : make_uint4(0u, 0u, 0u, 0u);
                        k += step_row, e += step_at;
                        if (e >= pieces) e -= pieces, ++k;
                    }
            }
            if (kb + PTA_PAGE < k1) fetch(kb + PTA_PAGE);
            __syncthreads();
            // scores of this wave's sixteen keys: element i is key 16 wave + 4 g + i, column r16
            ld_f32x4 sc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            const bf16_t* kr = Ks + (16 * wave + r16) * P + g * 8;
            const bf16_t* qr = Qs + r16 * P + g * 8;
            auto step = [&](ld_f32x4& sum, int c) {
                LdFrag k, q;
                k.u = *(const uint4*)(kr + 32 * c);
                q.u = *(const uint4*)(qr + 32 * c);
                sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k.v, q.v, sum, 0, 0, 0);
            };
            // The even pieces' sum and the odd ones', each by its own name.  Told apart by an index they kept the loop one step long, and a step took
            // 670 cycles (the sum moved in and out of place, a trip to LDS and back): 12,000 of the launch's 25,700 went there, and 1,600 go now (18 pieces).
            // With latent_values, 16 heads, R = 512, dr = 64: 8 sequences of 64 to 700 keys 17.8 -> 13.1 us, 2 of 1,900 19.4 -> 14.7, 16 of 4,000 48.0 -> 29.7.
#pragma unroll 3
            for (int c = 0; c + 1 < D / 32; c += 2) step(sc[0], c), step(sc[1], c + 1);
            if (D / 32 % 2) step(sc[0], D / 32 - 1);
            float p[4], top = -INFINITY;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                p[i] = kb + 16 * wave + 4 * g + i < k1 ? sc[0][i] + sc[1][i] : -INFINITY;
                top = fmaxf(top, p[i]);
            }
            top = column_max(top);
            if (g == 0) stat[wave * 16 + r16] = top;
            __syncthreads();
            const float m_new = fmaxf(fmaxf(fmaxf(stat[r16], stat[16 + r16]), fmaxf(stat[32 + r16], stat[48 + r16])), m_run);
            const float base = m_new == -INFINITY ? 0.f : m_new;
            const float corr = expf(m_run - base);
            float sum = 0.f;
            union { uint2 u; bf16_t b[4]; } w;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                w.b[i] = f32_to_bf16_bits(p[i] == -INFINITY ? 0.f : expf(p[i] - base));
                sum += bf16_bits_to_f32(w.b[i]);  // the weights as they were rounded
            }
            *(uint2*)(Ps + r16 * 72 + 16 * wave + 4 * g) = w.u;
            sum = column_sum(sum);
            if (g == 0) stat[64 + wave * 16 + r16] = sum;
            __syncthreads();
            l_run = l_run * corr + (stat[64 + r16] + stat[80 + r16] + stat[96 + r16] + stat[112 + r16]);
            m_run = m_new;
            LdFrag pf[2];
            pf[0].u = *(const uint4*)(Ps + r16 * 72 + g * 8);
            pf[1].u = *(const uint4*)(Ps + r16 * 72 + 32 + g * 8);
#pragma unroll
            for (int i = 0; i < TILES; ++i) {
                // by the transposing read: sixteen lanes give the addresses of four rows of sixteen elements and get an element of
                // the four rows each, lanes g keys 8 g .. + 3, then + 4 .. + 7 (R is whole tiles; one past it reads the last again)
                const bf16_t* vr = Ks + (g * 8 + (r16 >> 2)) * P + min((wave * TILES + i) * 16, R - 16) + (r16 & 3) * 4;
                LdFrag v[2];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e >> 1].half[e & 1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) ld_i16x4*)(vr + ((e >> 1) * 32 + (e & 1) * 4) * P));
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][e] *= corr;
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[0].v, pf[0].v, acc[i], 0, 0, 0);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[1].v, pf[1].v, acc[i], 0, 0, 0);
            }
        }
    }
    if (!there) return;
    const long at = row * splits + split;
    if (wave == 0 && g == 0) pm[at] = m_run, pl[at] = l_run;
    if (k0 >= k1) return;  // (its maximum says so: nothing else of it is read)
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
        const int el = (wave * TILES + i) * 16 + 4 * g;
        if (el < R) *(ld_f32x4*)(po + at * R + el) = acc[i];
    }
}

// ---- values -------------------------------------------------------------------------------------------------------------
// A workgroup has 32 outputs of one head for TOK tokens (fewer tokens a workgroup where there are few: what it reads is the
// ranges' sums, and one compute unit pulls some 24 GB/s): the ranges merged into LDS, then the product with 32 rows of the
// value expansion [H][V][R], two tiles of sixteen rows over two halves of R.  It is a chain of round trips: the expansion's rows are
// asked for before anything else, and LV_AHEAD ranges' sums at once (2 sequences of 1,900 keys, 30 ranges, 16 heads: 14.8 -> 8.1 us
// against four at once behind a branch each; 8 sequences of 64 to 700: 8.0 -> 6.8).
#define LV_SPLITS 1024
#define LV_STEPS 8   // of 32 elements, half of a latent of 512
#define LV_AHEAD 16

template <int TOK>
__global__ __launch_bounds__(256) void latent_values_kernel(const bf16_t* __restrict__ up_v, const float* __restrict__ pm, const float* __restrict__ pl,
                                                            const float* __restrict__ po, int M, int H, int R, int V, int splits, bf16_t* __restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) bf16_t lat[];  // [TOK][R + 8], then weights [TOK][splits]
    const int P = R + 8, h = blockIdx.x, v0 = blockIdx.y * 32, m0 = blockIdx.z * TOK;
    float* w_s = (float*)(lat + TOK * P);
    __shared__ ld_f32x4 part[2][64];
    __shared__ int live[TOK];  // ranges of a token that hold sums: those before the sequence's end
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    // the wave's rows of the expansion are on their way while the ranges are merged
    const int tile = wave & 1, half = wave >> 1, steps = R / 32;
    const int c0 = half ? (steps + 1) / 2 : 0, c1 = half ? steps : (steps + 1) / 2;
    const bf16_t* wr = up_v + ((long)h * V + min(v0 + 16 * tile + r16, V - 1)) * R + g * 8;
    LdFrag w[LV_STEPS];
#pragma unroll
    for (int c = 0; c < LV_STEPS; ++c) w[c].u = *(const uint4*)(wr + 32 * min(c0 + c, steps - 1));
    // a wave a token: e^(m_s - max) / sum
    for (int t = wave; t < TOK; t += 4) {
        const long row = (long)min(m0 + t, M - 1) * H + h;
        if (splits <= 64) {  // a lane a range: both of its numbers in one trip
            const int at = min(lane, splits - 1);
            const float l = pl[row * splits + at], any = pm[row * splits + at], m = lane < splits ? any : -INFINITY;
            const float top = wave_max(m), e = m == -INFINITY ? 0.f : expf(m - top), sum = wave_sum(e * l);
            const int last = (int)wave_max(m == -INFINITY ? 0.f : (float)(lane + 1));
            if (lane == 0) live[t] = last;
            if (lane < splits) w_s[t * splits + lane] = e * (1.0f / sum);
            continue;
        }
        float top = -INFINITY, sum = 0.f;
        int last = 0;
        for (int s = lane; s < splits; s += 64) {
            const float m = pm[row * splits + s];
            top = fmaxf(top, m);
            if (m != -INFINITY) last = s + 1;
        }
        top = wave_max(top);
        last = (int)wave_max((float)last);
        if (lane == 0) live[t] = last;
        for (int s = lane; s < splits; s += 64) {
            const float m = pm[row * splits + s], e = m == -INFINITY ? 0.f : expf(m - top);
            w_s[t * splits + s] = e;
            sum += e * pl[row * splits + s];
        }
        sum = wave_sum(sum);
        for (int s = lane; s < splits; s += 64) w_s[t * splits + s] *= 1.0f / sum;
    }
    __syncthreads();
    const int quads = R / 4;
    for (int i = tid; i < TOK * quads; i += 256) {
        const int t = i / quads, el = (i - t * quads) * 4, n = live[t];
        const long row = (long)min(m0 + t, M - 1) * H + h;
        const float* src = po + row * splits * R + el;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int s0 = 0; s0 < n; s0 += LV_AHEAD) {  // so many ranges' sums on their way at once
            float4 v[LV_AHEAD];
#pragma unroll
            for (int u = 0; u < LV_AHEAD; ++u) v[u] = *(const float4*)(src + (long)min(s0 + u, n - 1) * R);
#pragma unroll
            for (int u = 0; u < LV_AHEAD; ++u) {
                const float e = s0 + u < n ? w_s[t * splits + s0 + u] : 0.f;
                if (e == 0.f) continue;  // (a range whose keys weigh nothing)
                acc.x += e * v[u].x, acc.y += e * v[u].y, acc.z += e * v[u].z, acc.w += e * v[u].w;
            }
        }
        union { uint2 u; bf16_t b[4]; } o;
        o.b[0] = f32_to_bf16_bits(acc.x), o.b[1] = f32_to_bf16_bits(acc.y), o.b[2] = f32_to_bf16_bits(acc.z), o.b[3] = f32_to_bf16_bits(acc.w);
        *(uint2*)(lat + t * P + el) = o.u;
    }
    __syncthreads();
    const bf16_t* lr = lat + (r16 % TOK) * P + g * 8;
    ld_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < LV_STEPS; ++c) {
        if (c0 + c >= c1) break;
        LdFrag l;
        l.u = *(const uint4*)(lr + 32 * (c0 + c));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[c].v, l.v, acc, 0, 0, 0);
    }
    if (half) part[tile][lane] = acc;
    __syncthreads();
    if (half) return;
    const ld_f32x4 other = part[tile][lane];
    const int m = m0 + r16, v = v0 + 16 * tile + 4 * g;
    if (r16 >= TOK || m >= M) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (v + i < V) out[((long)m * H + h) * V + v + i] = f32_to_bf16_bits(acc[i] + other[i]);
}

// 1 if the decode launches take these sizes: rows and latents of whole pieces of 32, up to 512 elements of latent, plain
// queries of up to 256
extern "C" int pta_latent_decode_ok(int H, int dn, int dr, int R, int V) {
    return H > 0 && H <= 65535 && V > 0 && dn > 0 && dn % 32 == 0 && dn <= 256 && R > 0 && R % 32 == 0 && R <= 512 && dr >= 0 && dr % 8 == 0 &&
           (R + dr) % 32 == 0 && R + dr <= 640;
}

static const char* latent_shape_problem(int M, int H, int dn, int dr, int R, int V) {
    if (M <= 0 || M > 65535) return "tokens outside 1..65535";
    if (!pta_latent_decode_ok(H, dn, dr, R, V)) return "sizes that are not built";
    return nullptr;
}

extern "C" int pta_latent_queries(float* q_full, void* k_pool, const void* q_rows, long q_ld, const void* down_rows, long ld,
                                  const float* w_norm, float eps, const PtaRotation* rot, const int* token_pos, const int* token_seq,
                                  const int* block_table, int bt_stride, const void* kt, int M, int H, int dn, int dr, int R,
                                  int write_cache, void* stream) {
    if (const char* why = latent_shape_problem(M, H, dn, dr, R, 1)) return pta_fail("latent_queries: %s", why);
    PTA_REQUIRE(q_ld % 8 == 0 && (uintptr_t)q_rows % 16 == 0 && (uintptr_t)kt % 16 == 0 && (uintptr_t)q_full % 16 == 0,
                "latent_queries: queries and matrices must be sixteen-byte aligned");
    LatentToken t;
    if (latent_token_args("latent_queries", t, q_full, k_pool, q_rows, q_ld, down_rows, ld, w_norm, eps, rot, token_pos, token_seq, block_table,
                          bt_stride, M, H, dn, dr, R, write_cache))
        return 1;
    PTA_REQUIRE(kt, "latent_queries: null pointer");
    const int expand = H * ((R + 63) / 64);
    const dim3 grid(expand + M + (write_cache ? M : 0));
    hipStream_t s = (hipStream_t)stream;
#define LQ(KC) \
    case KC: hipLaunchKernelGGL(latent_queries_kernel<KC>, grid, dim3(256), 0, s, q_full, (bf16_t*)k_pool, (const bf16_t*)q_rows, q_ld, \
                                (const bf16_t*)kt, t, M, expand); break;
    switch (dn / 32) { LQ(1) LQ(2) LQ(3) LQ(4) LQ(5) LQ(6) LQ(7) LQ(8) }
#undef LQ
    return pta_check_launch("latent_queries");
}

extern "C" int pta_latent_decode(void* out, float* po, float* pm, float* pl, const float* q, const void* k_pool, const int* block_table,
                                 int bt_stride, const int* seq_start, const void* up_v, int M, int H, int R, int dr, int V, float scale,
                                 int size, int splits, void* stream) {
    if (const char* why = latent_shape_problem(M, H, 32, dr, R, V)) return pta_fail("latent_decode: %s", why);
    PTA_REQUIRE(out && po && pm && pl && q && k_pool && block_table && seq_start && up_v, "latent_decode: null pointer");
    PTA_REQUIRE(size > 0 && size % PTA_PAGE == 0 && splits >= 1 && splits <= LV_SPLITS, "latent_decode: %d ranges of %d keys", splits, size);
    PTA_REQUIRE((((uintptr_t)po | (uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)up_v) % 16) == 0, "latent_decode: pointers must be sixteen-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const int D = R + dr;
    const size_t lds = (size_t)(80 * (D + 8) + 16 * 72) * sizeof(bf16_t) + 128 * sizeof(float);
    const dim3 grid((H + 15) / 16, splits, M);
#define LP(T) do { \
        static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(latent_pages_kernel<T>), \
                                                             hipFuncAttributeMaxDynamicSharedMemorySize, 112 * 1024); \
        PTA_REQUIRE(raised == hipSuccess, "latent_decode: %zu bytes of LDS were refused", lds); \
        hipLaunchKernelGGL(latent_pages_kernel<T>, grid, dim3(256), lds, s, q, (const bf16_t*)k_pool, block_table, seq_start, bt_stride, size, splits, H, D, R, \
                           scale, po, pm, pl); \
    } while (0)
    if (R <= 64) LP(1);
    else if (R <= 128) LP(2);
    else if (R <= 256) LP(4);
    else LP(8);
#undef LP
    if (pta_check_launch("latent_pages")) return 1;
    // two tokens a workgroup while that leaves the compute units fewer than two each, else four, then sixteen
    const int outs = H * ((V + 31) / 32);
    const int units = pta_compute_units();
    const int tok = (long)outs * ((M + 1) / 2) <= 2L * units ? 2 : (long)outs * ((M + 3) / 4) <= 4L * units ? 4 : 16;
    const dim3 vgrid(H, (V + 31) / 32, (M + tok - 1) / tok);
    const size_t vlds = (size_t)tok * ((R + 8) * sizeof(bf16_t) + splits * sizeof(float));
#define LV(T) do { \
        static const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(latent_values_kernel<T>), \
                                                             hipFuncAttributeMaxDynamicSharedMemorySize, 112 * 1024); \
        PTA_REQUIRE(raised == hipSuccess, "latent_decode: %zu bytes of LDS were refused", vlds); \
        hipLaunchKernelGGL(latent_values_kernel<T>, vgrid, dim3(256), vlds, s, (const bf16_t*)up_v, pm, pl, po, M, H, R, V, splits, (bf16_t*)out); \
    } while (0)
    if (tok == 2) LV(2);
    else if (tok == 4) LV(4);
    else LV(16);
#undef LV
    return pta_check_launch("latent_values");
}
