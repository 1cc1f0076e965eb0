// C[M,N] = act(A[M,K] . W[N,K]^T + bias) + add1 + add2 in 32-bit, on the bfloat16 matrix instruction.
// The 32-bit path of the whole model runs its projections, feed-forwards and output head through here.
//
// A value times 2^16 is the sum of three bfloat16 values, exactly: the nearest one, the nearest one to what is left, and the rest,
// which has at most eight bits (split8).  (Without the factor the parts of values under 2^-110 would fall below bfloat16's smallest, 2^-133.
// With it those of the smallest value, 2^-149, do not.)  Of the nine products of the parts of two values six are formed, each exact in
// 32 bits.  The three left out, next times rest twice and rest times rest, come to 2^-24 of the product of the values at most, 2^-27.4 in
// the root of the mean square.  Six instructions of 16 cycles take the place of eight of 32 (v_mfma_f32_16x16x4_f32, 154 TFLOP/s).
//
// A value of 2^111 and more, infinite or undefined, has no such parts and leaves the sums it takes part in undefined; sums of 2^96 and more
// leave the range.  Those, and all with K under SHORT_K, are formed on the 32-bit instruction (whole_sum); all others stay as they
// are.
//
// Order of summation.  A row's result is bitwise the same alone and in any batch, so every kernel here sums the products
// of an output in one order, which K alone decides: K is walked in blocks of 32 elements (the last one filled up with
// zeros), the blocks are cut into up to eight segments of equal length, a segment is one chain of matrix instructions
// (a block is six of them, the smallest parts first), and the segments' sums are added in order.  Where a row lies in
// the grid, which kernel runs and how many workgroups share the segments changes nothing.
//
// The error against 64 bits, relative to the root of the sum of a row's squared products, in units of 2^-24 (rms): 0.8 at K = 64,
// 3.1 at 1,040, 6.2 at 4,544 and 13.4 at 18,176.  Chains of the 32-bit instruction over the same segments gave 1.4, 3.7, 7.2 and
// 14.3: an instruction here adds 32 products at a time, so a chain has fewer roundings.
//
// Measured against the 32-bit instruction, microseconds: 2,053 rows by 4,544 x 4,544 703 -> 446 (190 TFLOP/s), by 18,176 x 4,544
// 2,632 -> 1,650 (205), by 4,544 x 18,176 2,787 -> 1,640 (207); 60 rows by the same 42 -> 33, 146 -> 94, 120 -> 103; one row 21.2
// -> 19.8, 71 -> 60, 65 -> 65, by 65,024 x 4,544 239 -> 198 (6.0 TB/s).  (The factor costs the tiles 4 %: 424, 1,620 and 1,570 us without.)
//
// Three ways to the same numbers, by what bounds them (few_rows, f32_plan):
//   few rows: every weight is read once and that is the time.
//   many rows: tiles through two LDS buffers, bound by the matrix cores and the chip's power (8,192 x 8,192 x 4,096: 58 to 62 % of
//     the cycles at 1.9 GHz).
//   too few tiles to fill the chip, or to fill its last round: the segments of a tile are shared out over workgroups, whose
//     sums go to memory and are added by a small launch.
#include "common.h"
#include "lds_stream.h"
#include "pta_kernels.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

#define SEGS 8          // segments of K, at most
#define BK 32           // elements of K of a block
#define MOST_SUMS (32L << 20)           // 32-bit values that the segments' sums of cut tiles may take
#define MOST_K (0x7f000000 / (256 * 4))  // elements of a row that tiles can address
#define TILE_GROUP 8    // tiles along A that stand side by side in the order of tiles

struct F32Epilogue {
    const float* bias;
    const float* add1;
    const float* add2;
    int act;
    int wide;  // rows of C, add1 and add2 are read and written sixteen bytes at a time
};

__device__ __forceinline__ float finish(float v, const F32Epilogue& e, int n, long at) {
    if (e.bias) v += e.bias[n];
    if (e.act) v = apply_act(v, e.act);
    if (e.add1) v += e.add1[at];
    if (e.add2) v += e.add2[at];
    return v;
}

// four neighbours of row m of C from column n on, as far as they lie before column `end`
__device__ __forceinline__ void store4(float* C, f32x4 v, const F32Epilogue& e, int m, int n, int end, int N) {
    const long at = (long)m * N + n;
    if (e.wide && n + 4 <= end) {
        if (e.bias) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] += e.bias[n + j];
        }
        if (e.act) {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = apply_act(v[j], e.act);
        }
        if (e.add1) v += *(const f32x4*)(e.add1 + at);
        if (e.add2) v += *(const f32x4*)(e.add2 + at);
        *(f32x4*)(C + at) = v;
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (n + j < end) C[at + j] = finish(v[j], e, n + j, at + j);
}

// How rows are read: element by element; sixteen bytes at a time (rows sixteen-byte aligned, K a multiple of 4); the same
// without a look at the end (K a multiple of 32, what every published size is).
enum RowLoads { ROW_ELEMENTS, ROW_VECTORS, ROW_WHOLE };

// four consecutive elements of a row from k on, zeros beyond K (ROW_WHOLE: k + 4 <= K is the caller's)
template <int ROWS>
__device__ __forceinline__ f32x4 load4(const float* row, int k, int K) {
    if (ROWS == ROW_WHOLE) return *(const f32x4*)(row + k);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (ROWS == ROW_VECTORS) {
        if (k < K) v = *(const f32x4*)(row + k);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (k + j < K) v[j] = row[k + j];
    }
    return v;
}

__host__ __device__ static inline int k_blocks(int K) { return (K + BK - 1) / BK; }
__host__ __device__ static inline int seg_blocks(int K) { return (k_blocks(K) + SEGS - 1) / SEGS; }
__host__ __device__ static inline int segments(int K) { return (k_blocks(K) + seg_blocks(K) - 1) / seg_blocks(K); }

// ---- the three parts of a value -------------------------------------------------------------------------------------------
#define SCALE 0x1p16f    // of both operands
#define UNSCALE 0x1p-32f  // of their sums

struct Parts {
    bf16x8 part[3];  // nearest, next, rest
};

typedef __bf16 bf16_pair __attribute__((ext_vector_type(2)));
union PairBits {
    bf16_pair h;
    uint32_t u;
};
// (kept from the compiler, which would give -1 below as an inline constant, and the instruction reads that as the 32-bit one)
__device__ __forceinline__ bf16_pair pair_in_register(uint32_t bits) {
    PairBits p;
    p.u = bits;
    asm("" : "+s"(p.u));
    return p.h;
}

// A lane's eight elements of a block: k from 4 c on and k from 16 + 4 c on, c = lane / 16 (any order will do that both
// operands have; this one reads 64 bytes of a row by four lanes).  DOT: what is left behind the first part is made by one instruction a
// value, the dot product of the two parts with (-1, 0) or (0, -1) added to the value (exact, as the subtraction is, which takes two).
// A wave of the few-row kernels has nothing to do meanwhile (18,176 elements a row, one row: 67.3 us, 64.7 so, 64.2 without
// the factor; for both parts 65.8); beside many matrix instructions it is the slower one (2,053 rows by 4,544 x 18,176 1,640 us, 1,930 so).
template <bool DOT>
__device__ __forceinline__ Parts split8(f32x4 a, f32x4 b) {
    typedef float f32_pair __attribute__((ext_vector_type(2)));
    const bf16_pair first = pair_in_register(0x0000bf80u), second = pair_in_register(0xbf800000u);
    union { bf16x8 v[3]; uint32_t u[3][4]; } out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float x = SCALE * (i < 2 ? a[2 * i] : b[2 * i - 4]), y = SCALE * (i < 2 ? a[2 * i + 1] : b[2 * i - 3]);
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            PairBits c;
            c.h = __builtin_convertvector(f32_pair{x, y}, bf16_pair);  // one instruction for the two
            out.u[p][i] = c.u;
            if (p == 0 && DOT) {
                x = __builtin_amdgcn_fdot2_f32_bf16(c.h, first, x, false);
                y = __builtin_amdgcn_fdot2_f32_bf16(c.h, second, y, false);
            } else if (p < 2) {
                x -= __uint_as_float(c.u << 16);
                y -= __uint_as_float(c.u & 0xffff0000u);
            }
        }
    }
    return Parts{{out.v[0], out.v[1], out.v[2]}};
}

// the six products, the smallest first
#define TERMS 6
__device__ constexpr int term_w(int t) { return t == 0 ? 2 : t < 3 ? 1 : 0; }
__device__ constexpr int term_x(int t) { return t == 3 ? 2 : t == 1 || t == 4 ? 1 : 0; }

// Products so short take the 32-bit instruction: what the six products of parts leave out is more than its roundings.  The error against 64
// bits in 2^-24 (rms), 32-bit instruction and parts, of normal values relative to the root of the sum of squared products / of values
// over ten orders of magnitude relative to the sum of absolute products: K = 1 0.42 / 0.42 and 0.58 / 0.58, 2 0.53 / 0.49 and 0.56 / 0.57, 4
// 0.67 / 0.60 and 0.53 / 0.61, 5 0.74 / 0.64 and 0.57 / 0.64, 6 0.79 / 0.69 and 0.57 / 0.64, 8 0.91 / 0.76 and 0.56 / 0.65.
#define SHORT_K 6

// The sums of sixteen rows of W from n on by sixteen of A from m on, from those of the parts; what of them is not finite, and all
// of a short K, as one chain over all of K on the 32-bit instruction.
template <int ROWS>
__device__ __forceinline__ f32x4 whole_sum(f32x4 v, const float* A, const float* W, int m, int n, int M, int N, int K) {
    bool out[4], any = false;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        out[e] = K < SHORT_K || !(fabsf(v[e]) <= 3.402823466e38f);
        any |= out[e];
        v[e] *= UNSCALE;
    }
    if (!__any(any)) return v;
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = 4 * (lane >> 4);
    const float* wr = W + (long)min(n + r16, N - 1) * K;
    const float* xr = A + (long)min(m + r16, M - 1) * K;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int k = kq; k < K + kq; k += 16) {
        const f32x4 w = load4<ROWS == ROW_WHOLE ? ROW_VECTORS : ROWS>(wr, k, K), x = load4<ROWS == ROW_WHOLE ? ROW_VECTORS : ROWS>(xr, k, K);
#pragma unroll
        for (int j = 3; j >= 0; --j) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], sum, 0, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (out[e]) v[e] = sum[e];
    return v;
}

// ---- few rows ---------------------------------------------------------------------------------------------------------
// Every weight is read once and that is the time.  A workgroup owns up to 32 rows of W and its eight waves a segment each; W
// goes from memory into registers, its parts into the instruction's operands, the sums meet in LDS.
// CT: tiles of sixteen rows of A, RT: tiles of sixteen rows of W.  D blocks of K are asked for while the D before them are
// multiplied: at K = 4,544 and one row of A a compute unit then has some 60 KB on its way.  What is asked for past a segment's
// end is its last block again, which a cache has (the next segment's first blocks, long gone from the caches, were a sixth of all
// that came from memory at 4,544 x 4,544; the launch takes 22 us either way).
template <int CT, int RT, int D, int ROWS>
__global__ __launch_bounds__(512, CT * RT <= 2 ? 2 : 1) void gemm_f32_few_kernel(
    float* __restrict__ C, const float* __restrict__ A, const float* __restrict__ W, F32Epilogue epi, int M, int N, int K) {
    __shared__ f32x4 part[SEGS][RT * CT][64];
    const int lane = threadIdx.x & 63, seg = threadIdx.x >> 6;
    const int r16 = lane & 15, kq = 4 * (lane >> 4);
    // the rows of W are shared out evenly: a launch takes as long as the compute unit with the most of them
    const int n0 = (int)((long)blockIdx.x * N / gridDim.x), n1 = (int)((long)(blockIdx.x + 1) * N / gridDim.x);
    const int nb = k_blocks(K), sb = seg_blocks(K);
    const int b0 = seg * sb, b1 = min(nb, b0 + sb);
    const float* wr[RT];
    const float* xr[CT];
#pragma unroll
    for (int r = 0; r < RT; ++r) wr[r] = W + (long)min(n0 + 16 * r + r16, n1 - 1) * K;  // rows past the end: read again, not kept
#pragma unroll
    for (int c = 0; c < CT; ++c) xr[c] = A + (long)min(16 * c + r16, M - 1) * K;
    f32x4 acc[RT][CT];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 w[2][D][RT][2], x[2][D][CT][2];
    auto fetch = [&](int buf, int b) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const int k = BK * min(b + i, b1 - 1) + kq;  // past the segment: its last block again, not used
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int r = 0; r < RT; ++r) w[buf][i][r][h] = load4<ROWS>(wr[r], k + 16 * h, K);
#pragma unroll
                for (int c = 0; c < CT; ++c) x[buf][i][c][h] = load4<ROWS>(xr[c], k + 16 * h, K);
            }
        }
    };
    auto multiply = [&](int buf, int b) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            if (b + i < b1) {
                Parts xs[CT];
#pragma unroll
                for (int c = 0; c < CT; ++c) xs[c] = split8<true>(x[buf][i][c][0], x[buf][i][c][1]);
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    const Parts ws = split8<true>(w[buf][i][r][0], w[buf][i][r][1]);
#pragma unroll
                    for (int t = 0; t < TERMS; ++t)
#pragma unroll
                        for (int c = 0; c < CT; ++c)
                            acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws.part[term_w(t)], xs[c].part[term_x(t)], acc[r][c], 0, 0, 0);
                }
            }
        }
    };
    if (b0 < b1) {
        fetch(0, b0);
        for (int b = b0; b < b1; b += 2 * D) {
            fetch(1, b + D);
            multiply(0, b);
            fetch(0, b + 2 * D);
            multiply(1, b + D);
        }
    }
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c) part[seg][r * CT + c][lane] = acc[r][c];
    __syncthreads();
    const int used = (nb + sb - 1) / sb;
    for (int i = threadIdx.x; i < RT * CT * 64; i += 512) {
        const int t = i >> 6, l = i & 63;  // a wave has a tile
        f32x4 v = part[0][t][l];
        for (int s = 1; s < used; ++s) v += part[s][t][l];
        v = whole_sum<ROWS>(v, A, W, 16 * (t % CT), n0 + 16 * (t / CT), M, N, K);
        const int m = 16 * (t % CT) + (l & 15);
        const int n = n0 + 16 * (t / CT) + 4 * (l >> 4);
        if (m < M) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (n + j < n1) C[(long)m * N + n + j] = finish(v[j], epi, n + j, (long)m * N + n + j);
        }
    }
}

// The same for up to sixteen rows of A where rows are sixteen-byte aligned: rows of W straight to LDS in whole lines (lds_stream.h),
// D blocks ahead, a wave's segment at a time, and on to the workgroup's next rows without a pause: a workgroup has all the rows of W of a
// compute unit, in tiles of up to 16 RT.  Sums change hands through LDS, in two places in turn, one barrier a tile.
// 18,176 x 4,544, us with registers and three rounds of workgroups -> this: 1 row 70.0 -> 60.5 (5.5 TB/s), 16 rows 86.5 -> 67; 4,544 x
// 18,176 67 -> 65, 83 -> 70; 32,768 x 2,048 59.9 -> 53.9, 72.3 -> 55.6.
//
// Two products of the same rows of A in one launch (PRODUCTS 2: a block's query_key_value and first feed-forward matrix, or the last
// matrices of both branches, whose K and A differ): a workgroup has its share of the rows of both and its rings go on from the first to the
// second as from tile to tile, so that one launch starts and ends where two did.  With `add_first` (matrices of one N) the first's
// results, bias and activation done, lie in LDS until the second's have them added.  us on their own -> so, 1 / 8 / 16 rows: 4,672 and 18,176 by
// 4,544 85.4 -> 80.4, 90.7 -> 85.5, 95.5 -> 90.7; 4,544 by 4,544 and by 18,176 95.6 -> 87.7, 94.7 -> 85.7, 97.2 -> 89.3; 2,048 by 2,048
// and by 8,192 33.8 -> 31.7, 36.9 -> 31.8, 37.7 -> 32.9; 3,072 and 4,096 by 1,024 14.2 -> 11.7, 13.4 -> 11.7, 13.5 -> 11.9.  Of the
// 80.4 some 73 are the loads; taking values apart is not all hidden beside them (a third block on its way changed nothing).
template <int RT, int D>
struct FewRing {
    static constexpr int SLOT = (RT + 1) * 2048, RING = D * SLOT, LOADS = 2 * (RT + 1);
    static constexpr int LDS = SEGS * RING + 2 * SEGS * RT * 1024;
};

struct F32Few {
    float* C;
    const float* A;
    const float* W;
    F32Epilogue epi;
    int N, K;
    int each, over;  // rows of W a workgroup has, and how many of the first workgroups have one more
};

template <int PRODUCTS>
struct F32FewJob {
    F32Few of[PRODUCTS];
};

template <int RT, int D, int PRODUCTS>
__global__ __launch_bounds__(512, 2) void gemm_f32_few_ring_kernel(F32FewJob<PRODUCTS> job, int M, int add_first) {
    using R = FewRing<RT, D>;
    extern __shared__ __attribute__((aligned(1024))) char lds[];  // the waves' rings, the sums, [2][segment][RT][64], the first's results
    const int lane = threadIdx.x & 63, seg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    char* ring = lds + seg * R::RING;
    f32x4* sums = reinterpret_cast<f32x4*>(lds + SEGS * R::RING);
    float* kept = reinterpret_cast<float*>(lds + R::LDS);  // [row of the workgroup][16]
    const unsigned to = __builtin_amdgcn_readfirstlane(lds_address(ring));
    const int c4[2] = {stream_element(lane, 0) / 2, stream_element(lane, 1) / 2};  // four values where a bfloat16 row has eight
    struct Mine {  // what a workgroup, and of its K this wave, has of a product
        int n0, rows, tiles, per_tile, b0, blocks;
    };
    auto mine_of = [&](const F32Few& p) {
        Mine m;
        m.n0 = blockIdx.x * p.each + min((int)blockIdx.x, p.over);
        m.rows = p.each + ((int)blockIdx.x < p.over ? 1 : 0);
        m.tiles = max((m.rows + 16 * RT - 1) / (16 * RT), 1);
        m.per_tile = (m.rows + m.tiles - 1) / m.tiles;
        m.b0 = seg * seg_blocks(p.K);
        m.blocks = max(min(k_blocks(p.K) - m.b0, seg_blocks(p.K)), 1);  // (a wave without a segment multiplies a block of zeros)
        return m;
    };
    // what is asked for next: a block of a tile of a product
    const float *w_from, *x_from;
    int w_bytes, x_bytes;
    Mine next;
    int K, product = -1, tile = 0, block = 0, row_at[R::LOADS];  // rows of W, and of A behind them
    auto rows_of = [&]() {
#pragma unroll
        for (int l = 0; l < 2 * RT; ++l) {
            const int i = (l >> 1) * 16 + stream_row(lane, l & 1), row = tile * next.per_tile + i;
            row_at[l] = i < next.per_tile && row < next.rows ? row * K * 4 : LDS_PAST;
        }
    };
    auto next_product = [&]() {
        if (++product == PRODUCTS) return;
        const F32Few& p = job.of[product];
        next = mine_of(p);
        K = p.K;
        w_from = p.W + (long)next.n0 * K, w_bytes = next.rows * K * 4;
        x_from = p.A, x_bytes = M * K * 4;
        tile = block = 0;
        rows_of();
#pragma unroll
        for (int l = 0; l < 2; ++l) row_at[2 * RT + l] = stream_row(lane, l) < M ? stream_row(lane, l) * K * 4 : LDS_PAST;
    };
    auto issue = [&](int slot) {
        const i32x4_t w = buffer_of(w_from, w_bytes), x = buffer_of(x_from, x_bytes);
        const int k = product < PRODUCTS ? (next.b0 + block) * BK : K;
#pragma unroll
        for (int l = 0; l < R::LOADS; ++l)
            fetch16(l < 2 * RT ? w : x, to + slot + l * 1024, row_at[l] != LDS_PAST && k + c4[l & 1] < K ? row_at[l] + (k + c4[l & 1]) * 4 : LDS_PAST);
        if (product < PRODUCTS && ++block == next.blocks) {
            block = 0;
            if (++tile < next.tiles) rows_of();
            else next_product();
        }
    };
    next_product();
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d * R::SLOT);
    const int in_row = r16 * 128 + ((g ^ (r16 >> 1)) & 7) * 16;  // elements 4 g of a block, and 64 flipped 16 + 4 g
    int slot = 0, turn = 0;  // tiles so far, of both products
#pragma unroll 1
    for (int q = 0; q < PRODUCTS; ++q) {
        const F32Few& p = job.of[q];
        const Mine mine = mine_of(p);
        const int used = segments(p.K);
        for (int t = 0; t < mine.tiles; ++t, ++turn) {
            f32x4 acc[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) acc[r] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int b = 0; b < mine.blocks; ++b) {
                wait_loads<(D - 1) * R::LOADS>();
                f32x4 v[RT + 1][2];
#pragma unroll
                for (int r = 0; r <= RT; ++r)
#pragma unroll
                    for (int h = 0; h < 2; ++h) v[r][h] = *reinterpret_cast<const f32x4*>(ring + ((in_row ^ (h * 64)) + slot + r * 2048));
                wait_reads();
                __builtin_amdgcn_sched_barrier(0);
                issue(slot);  // into the slot just read
                __builtin_amdgcn_sched_barrier(0);
                const Parts xs = split8<true>(v[RT][0], v[RT][1]);
#pragma unroll
                for (int r = 0; r < RT; ++r) {
                    const Parts ws = split8<true>(v[r][0], v[r][1]);
#pragma unroll
                    for (int term = 0; term < TERMS; ++term)
                        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws.part[term_w(term)], xs.part[term_x(term)], acc[r], 0, 0, 0);
                }
                slot = slot == R::RING - R::SLOT ? 0 : slot + R::SLOT;
            }
            f32x4* meet_at = sums + (turn & 1) * (SEGS * RT * 64);
#pragma unroll
            for (int r = 0; r < RT; ++r) meet_at[(seg * RT + r) * 64 + lane] = acc[r];
            wait_reads();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const int r = (seg - turn * RT) & (SEGS - 1);  // the waves take turns at what follows
            if (r >= RT) continue;
            f32x4 u = meet_at[r * 64 + lane];
            for (int s = 1; s < used; ++s) u += meet_at[(s * RT + r) * 64 + lane];
            const int end = min(mine.rows, (t + 1) * mine.per_tile), at16 = t * mine.per_tile + 16 * r;
            u = whole_sum<ROW_VECTORS>(u, p.A, p.W, 0, mine.n0 + at16, M, p.N, p.K);
            const bool keep = PRODUCTS > 1 && q == 0 && add_first;
            if (r16 < M) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int i = at16 + 4 * g + j, n = mine.n0 + i;  // (read a barrier and more after it was kept)
                    if (i >= end) continue;
                    if (PRODUCTS > 1 && q == 1 && add_first) {
                        F32Epilogue bare = p.epi;
                        bare.add1 = bare.add2 = nullptr;
                        const float v = finish(u[j], bare, n, 0) + kept[i * 16 + r16];
                        p.C[(long)r16 * p.N + n] = p.epi.add1 ? v + p.epi.add1[(long)r16 * p.N + n] : v;
                    } else {
                        const float v = finish(u[j], p.epi, n, (long)r16 * p.N + n);
                        if (keep) kept[i * 16 + r16] = v;
                        else p.C[(long)r16 * p.N + n] = v;
                    }
                }
            }
        }
    }
    wait_loads<0>();  // nothing is on its way to LDS any more
}

// ---- many rows ----------------------------------------------------------------------------------------------------------
// A workgroup of eight waves (four along the rows of W, two along the rows of A) makes a tile of 64 FP rows of W by 32 FQ rows
// of A, a block of K at a time.  Values come through registers, are taken apart once for the workgroup and lie in LDS as
// three planes of rows of 64 bytes, sixteen bytes c of row r at place c ^ (-(r / 4) % 4), so that any sixteen lanes that read
// together cover every bank once (they are not sixteen neighbours: with c ^ (r / 4 % 4) a third of the cycles were conflicts).  Two buffers, one barrier a block:
//
//   columns j = 0 .. FQ - 2: the parts of column j + 1 being read, a share of block b + 1 taken apart into the other buffer,
//                            block b + 2 asked for
//   barrier: the other buffer is whole, and everyone has read this one
//   column FQ - 1: the next block's parts being read as those of this block have been used
struct F32Tiles {
    float* C;
    float* part;  // segments' sums of cut tiles: [segment][tile][wave][fragment][lane][4]
    const float* A;
    const float* W;
    int M, N, K;
    int tiles_q, tiles_p;  // tiles along the rows of A and of W
    int whole;             // the first tiles, computed over all of K
    int share;             // workgroups that share the segments of each of the others
};

__device__ __forceinline__ void tile_at(const F32Tiles& job, int t, int& tp, int& tq) {
    const int per_group = TILE_GROUP * job.tiles_p;
    const int grp = t / per_group, in = t - grp * per_group;
    const int width = min(TILE_GROUP, job.tiles_q - grp * TILE_GROUP);
    tp = in / width;
    tq = grp * TILE_GROUP + in - tp * width;
}

__device__ __forceinline__ void meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads and writes of LDS are done
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

#define PAST 0x7f000000  // an offset past the end of every tile's rows: such loads give zeros

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const float* p, long values) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(values * 4), 0x00020000);
}

static constexpr __host__ __device__ int lds_bytes(int FP, int FQ) { return 2 * 3 * (64 * FP + 32 * FQ) * 64; }

template <int FP, int FQ, int ROWS>
__global__ __launch_bounds__(512, 2) void gemm_f32_tile_kernel(F32Tiles job, F32Epilogue epi) {
    static_assert(lds_bytes(FP, FQ) <= 160 * 1024 && FP * FQ * 8192 <= lds_bytes(FP, FQ), "the blocks and the sums must fit LDS");
    constexpr int TP = 64 * FP, TQ = 32 * FQ, PLANE = (TP + TQ) * 64, BUF = 3 * PLANE, IP = FP / 2;
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, c4 = lane >> 4, wp = wave & 3, wq = wave >> 2;
    const int M = job.M, N = job.N, K = job.K;
    const int tiles = job.tiles_p * job.tiles_q, nb = k_blocks(K), sb = seg_blocks(K), used = segments(K);
    // which tile, which segments: workgroups go to the eight dies in turn, each die takes a run of tiles
    int t, s0 = 0, s1 = used, rest = -1;
    const int whole8 = (job.whole + 7) >> 3;
    if ((int)blockIdx.x < whole8 * 8) {
        t = (blockIdx.x & 7) * whole8 + (blockIdx.x >> 3);
        if (t >= job.whole) return;
    } else {
        const int R = tiles - job.whole, all = R * job.share, per = (all + 7) >> 3;
        const int i = blockIdx.x - whole8 * 8, at = (i & 7) * per + (i >> 3);
        if (at >= all) return;
        const int range = at / R;
        rest = at - range * R;
        t = job.whole + rest;
        s0 = range * used / job.share;
        s1 = (range + 1) * used / job.share;
    }
    int tp, tq;
    tile_at(job, t, tp, tq);
    const int n0 = tp * TP, m0 = tq * TQ;
    const int b0 = s0 * sb, b1 = min(nb, s1 * sb);

    // What a thread brings of a block: eight elements of IP rows of W and, in the first 2 FQ waves, of a row of A.  Rows past the
    // last one lie past the buffer's end and give zeros, as do elements past K.
    const int row = threadIdx.x >> 2, kq = 4 * (threadIdx.x & 3);
    const bool has_x = wave < 2 * FQ;
    const __amdgpu_buffer_rsrc_t rw = buffer_of(job.W + (long)n0 * K, (long)min(TP, N - n0) * K);
    const __amdgpu_buffer_rsrc_t rx = buffer_of(job.A + (long)m0 * K, (long)min(TQ, M - m0) * K);
    const int at_row = (row * K + kq) * 4;
    const int to = row * 64 + (((threadIdx.x & 3) ^ (-(row >> 2) & 3)) * 16);
    f32x4 v[IP + 1][2];
    auto fetch = [&](int i, int b) __attribute__((always_inline)) {
        if (i == IP && !has_x) return;
        const int k = BK * min(b, nb - 1);  // past the last block: that one again, not used
        const __amdgpu_buffer_rsrc_t from = i == IP ? rx : rw;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int at = at_row + (i == IP ? 0 : i * 512 * K);
            if (ROWS == ROW_ELEMENTS) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[i][h][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(from, k + kq + 16 * h + e < K ? at + 4 * e : PAST, (k + 16 * h) * 4, 0));
            } else {
                v[i][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, ROWS == ROW_WHOLE || k + kq + 16 * h < K ? at : PAST, (k + 16 * h) * 4, 0));
            }
        }
    };
    auto stage = [&](int i, int buf) __attribute__((always_inline)) {
        if (i == IP && !has_x) return;
        const Parts s = split8<false>(v[i][0], v[i][1]);
        char* at = lds + buf + (i == IP ? TP * 64 : i * 8192) + to;
#pragma unroll
        for (int p = 0; p < 3; ++p) *(bf16x8*)(at + p * PLANE) = s.part[p];
    };

    f32x4 acc[FP][FQ], total[FP][FQ];
#pragma unroll
    for (int i = 0; i < FP; ++i)
#pragma unroll
        for (int j = 0; j < FQ; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int in_row = r16 * 64 + ((c4 ^ (-(r16 >> 2) & 3)) * 16);
    const int at_w = wp * FP * 1024 + in_row, at_x = TP * 64 + wq * FQ * 1024 + in_row;
    bf16x8 w[FP][3], x[2][3];
    auto read_w = [&](int buf, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FP; ++i) w[i][p] = *(const bf16x8*)(lds + buf + p * PLANE + at_w + i * 1024);
    };
    auto read_x = [&](int buf, int j, int set) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 3; ++p) x[set][p] = *(const bf16x8*)(lds + buf + p * PLANE + at_x + j * 1024);
    };
    auto multiply = [&](int j, int set, int term) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < FP; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][term_w(term)], x[set][term_x(term)], acc[i][j], 0, 0, 0);
    };
    f32x4* out = nullptr;
    if (rest >= 0) out = reinterpret_cast<f32x4*>(job.part) + (((long)s0 * (tiles - job.whole) + rest) * 8 + wave) * (FP * FQ * 64) + lane;
    const long out_step = (long)(tiles - job.whole) * 8 * FP * FQ * 64;

    int left = sb, cur = 0;
    // a block; `set`: where column 0's parts are
    auto block = [&](int b, int set) __attribute__((always_inline)) {
        const int nxt = BUF - cur;
#pragma unroll
        for (int j = 0; j < FQ; ++j) {
            const int s = (set + j) & 1;
            __builtin_amdgcn_sched_barrier(0);
            if (j + 1 < FQ) read_x(cur, j + 1, s ^ 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i <= IP; ++i)
                if (i == j || (i > j && j >= FQ - 2)) {
                    if (FQ > 1 && j == FQ - 1) continue;
                    stage(i, nxt);
                    fetch(i, b + 2);
                }
            if (j == FQ - 1) {
                meet();
                read_x(nxt, 0, s ^ 1);
            }
            __builtin_amdgcn_s_setprio(1);  // whoever multiplies goes first: 4 % at 8,192 x 8,192 x 4,096
#pragma unroll
            for (int term = 0; term < TERMS; ++term) {
                multiply(j, s, term);
                if (j == FQ - 1 && (term == 0 || term == 2 || term == 5)) {
                    __builtin_amdgcn_sched_barrier(0);
                    read_w(nxt, term == 0 ? 2 : term == 2 ? 1 : 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            __builtin_amdgcn_s_setprio(0);
        }
        cur = nxt;
        if (--left == 0 || b + 1 == b1) {  // the segment ends: its sum joins the others in their order
            if (rest >= 0) {
#pragma unroll
                for (int j = 0; j < FQ; ++j)
#pragma unroll
                    for (int i = 0; i < FP; ++i) out[(j * FP + i) * 64] = acc[i][j];
                out += out_step;
            } else if (b < sb) {
#pragma unroll
                for (int i = 0; i < FP; ++i)
#pragma unroll
                    for (int j = 0; j < FQ; ++j) total[i][j] = acc[i][j];
            } else {
#pragma unroll
                for (int i = 0; i < FP; ++i)
#pragma unroll
                    for (int j = 0; j < FQ; ++j) total[i][j] += acc[i][j];
            }
#pragma unroll
            for (int i = 0; i < FP; ++i)
#pragma unroll
                for (int j = 0; j < FQ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            left = sb;
        }
    };
#pragma unroll
    for (int i = 0; i <= IP; ++i) fetch(i, b0);
#pragma unroll
    for (int i = 0; i <= IP; ++i) {
        stage(i, 0);
        fetch(i, b0 + 1);
    }
    meet();
    read_x(0, 0, 0);
    read_w(0, 2);
    read_w(0, 1);
    read_w(0, 0);
    if (FQ & 1) {
        for (int b = b0; b < b1; b += 2) {
            block(b, 0);
            if (b + 1 < b1) block(b + 1, 1);
        }
    } else {
        for (int b = b0; b < b1; ++b) block(b, 0);
    }
    if (rest >= 0) return;

    meet();  // everyone is past reading the last block: a wave's sums change hands through LDS, fragment by fragment
    f32x4* mine = reinterpret_cast<f32x4*>(lds) + wave * (FP * FQ * 64) + lane;
#pragma unroll
    for (int j = 0; j < FQ; ++j)
#pragma unroll
        for (int i = 0; i < FP; ++i) mine[(j * FP + i) * 64] = total[i][j];
#pragma unroll 1
    for (int f = 0; f < FP * FQ; ++f) {
        const int m16 = m0 + (wq * FQ + f / FP) * 16, n16 = n0 + (wp * FP + f % FP) * 16;
        f32x4 u = mine[f * 64];
        u = whole_sum<ROWS>(u, job.A, job.W, m16, n16, M, N, K);
        const int m = m16 + r16, n = n16 + 4 * c4;
        if (m < M && n < N) store4(job.C, u, epi, m, n, N, N);
    }
}

// the cut tiles: the segments' sums added in order, and the epilogue; a wave has a fragment
template <int FP, int FQ, int ROWS>
__global__ __launch_bounds__(256) void gemm_f32_add_kernel(F32Tiles job, F32Epilogue epi) {
    const int R = job.tiles_p * job.tiles_q - job.whole, used = segments(job.K);
    const int lane = threadIdx.x & 63, at = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int rest = at / (8 * FP * FQ), wave = at / (FP * FQ) % 8, j = at % (FP * FQ) / FP, i = at % FP;
    if (rest >= R) return;
    int tp, tq;
    tile_at(job, job.whole + rest, tp, tq);
    const f32x4* from = reinterpret_cast<const f32x4*>(job.part) + (long)at * 64 + lane;
    const long step = (long)R * 8 * FP * FQ * 64;
    f32x4 p[SEGS];
#pragma unroll
    for (int s = 0; s < SEGS; ++s) p[s] = from[min(s, used - 1) * step];
    f32x4 v = p[0];
#pragma unroll
    for (int s = 1; s < SEGS; ++s)
        if (s < used) v += p[s];
    const int m16 = tq * 32 * FQ + ((wave >> 2) * FQ + j) * 16, n16 = tp * 64 * FP + ((wave & 3) * FP + i) * 16;
    v = whole_sum<ROWS>(v, job.A, job.W, m16, n16, job.M, job.N, job.K);
    const int m = m16 + (lane & 15), n = n16 + 4 * (lane >> 4);
    if (m < job.M && n < job.N) store4(job.C, v, epi, m, n, job.N, job.N);
}

// How a product runs: few rows (fp = 0), or tiles of 64 fp rows of W by 32 fq rows of A, the first `whole` of them over all of
// K, the segments of each of the others shared out over `share` workgroups.  What a choice takes, in microseconds, is put
// together from measurements at K = 1,024, 4,096 and 8,192 (256 compute units, 64 to 1,024 tiles):
//   a block of 32 elements of K: `full` with a tile for every compute unit, `half` with a tile for at most half of them, `pair`
//     with two on a unit, where two fit (0: they do not);
//   a tile's start and end: `ends`, `cut` for a tile whose K is cut (the difference: tiles of 256 x 128 keep part of the segments'
//     sums in memory, which costs them 2.5 us a segment);
//   sums of cut tiles: 4.5 us for the second launch and 0.25 us a megabyte.
// The smallest sum wins.
struct F32Plan {
    int fp, fq, whole, share;
    double us;
};

struct F32Costs {
    double half, full, pair, ends, cut;
};
static const F32Costs costs[2][4] = {
    {{0.56, 0.57, 0.93, 6.0, 6.0}, {0.73, 0.77, 1.39, 7.4, 7.4}, {0.94, 1.01, 0.0, 8.8, 8.8}, {1.10, 1.23, 0.0, 10.5, 10.0}},
    {{0.92, 0.95, 0.0, 8.0, 8.0}, {1.19, 1.32, 0.0, 10.5, 10.5}, {1.52, 1.76, 0.0, 12.6, 12.0}, {1.84, 2.17, 0.0, 32.0, 12.5}},
};

// Which products the kernels for few rows have.  Measured, microseconds of few rows and of the best tiles:
//   N x K            1 row            8 rows           16 rows          17 rows          32 rows
//   1,024 x 1,024     7.3 /   9.9      7.5 /  10.0      7.7 /  10.0      8.5 /   9.8     10.4 /   9.8
//   4,096 x 1,024     7.6 /  11.9      7.6 /  12.0      7.8 /  12.1     10.4 /  12.2     12.1 /  11.9
//   2,048 x 2,048     8.4 /  12.4      9.0 /  12.6      9.2 /  12.6     12.9 /  12.8     16.5 /  12.9
//   4,544 x 4,544    19.6 /  25.9     21.2 /  25.9     21.5 /  26.3     31.6 /  26.3     36.8 /  26.8
//   18,176 x 4,544   60.5 /  76.4     63.0 /  76.6     66.9 /  77.5     98.0 /  77.5      116 /  79.3
//   32,768 x 2,048   53.9 /  61.6     55.4 /  61.9     55.6 /  62.7     80.2 /  63.5     90.3 /  64.3
//   65,024 x 4,544    199 /   198      206 /   199      217 /   200      297 /   200      344 /   203
// With a short K, whose segments are a block or two, rows up to 64: 256 x 512 33 rows 8.6 and 9.9, 64 rows 10.5 and 10.0.
// Tiles address a row by 32-bit offsets (MOST_K).
static bool few_rows(int M, int N, int K) {
    if (K > MOST_K) return true;
    if (K < 1024) return M <= 64;
    if (K < 2048) return M <= 32;
    return M <= 16 && (N < 32768 || K < 4096);
}

static F32Plan f32_plan(int M, int N, int K) {
    F32Plan best{0, 0, 0, 1, 1e30};
    if (few_rows(M, N, K)) return best;
    const int units = pta_compute_units(), used = segments(K), blocks = k_blocks(K);
    for (int fp = 2; fp <= 4; fp += 2)
        for (int fq = 1; fq <= 4; ++fq) {
            const F32Costs& c = costs[fp / 2 - 1][fq - 1];
            const long tiles = (long)((N + 64 * fp - 1) / (64 * fp)) * ((M + 32 * fq - 1) / (32 * fq));
            const long slots = c.pair > 0.0 ? 2 * units : units;
            // `groups` workgroups, each on b blocks of K
            auto time = [&](long groups, int b, double ends) {
                const double round = b * (c.pair > 0.0 ? c.pair : c.full) + ends;
                double us = (double)(groups / slots) * round;
                const long left = groups % slots;
                if (left > units) us += round;
                else if (left) us += b * (c.half + (c.full - c.half) * (left > units / 2 ? 2.0 * left / units - 1.0 : 0.0)) + ends;
                return us;
            };
            auto consider = [&](long whole, int share, double us) {
                if (us < best.us) best = F32Plan{fp, fq, (int)whole, share, us};
            };
            consider(tiles, 1, time(tiles, blocks, c.ends));
            const long left = tiles % slots;
            if (!left) continue;
            const double body = time(tiles - left, blocks, c.ends);
            for (int share = 2; share <= used; ++share) {
                const int each = (used + share - 1) / share * seg_blocks(K);  // of the workgroup with the most segments
                if (left * used * fp * fq * 2048 > MOST_SUMS) break;
                consider(tiles - left, share, body + time(left * share, each, c.cut) + 4.5 + 0.25 * left * used * fp * fq * 8192e-6);
            }
        }
    return best;
}

template <int ROWS>
static void launch_few(float* C, const float* A, const float* W, F32Epilogue epi, int rows, int N, int K, hipStream_t s) {
    // whole rounds of the compute units, up to 32 rows of W each; small matrices: four rows a workgroup
    const int all = pta_compute_units();
    int groups = all * ((N + all * 32 - 1) / (all * 32));
    if (groups > (N + 3) / 4) groups = (N + 3) / 4;
    const bool two = (N + groups - 1) / groups > 16;
    // Rings in LDS: their offsets are 32-bit bytes within a workgroup's rows.  Up to sixteen rows of W a unit, whose waves take a block
    // or two each, they pay from five rows of A on: 2,048 x 2,048 1 row 7.9 us, in rings 8.7, 8 rows 9.6 and 8.8, 16 rows 11.1 and 8.9.
    const int units = groups < all ? groups : all;  // one workgroup a unit, with its rows of all rounds
    if (ROWS != ROW_ELEMENTS && rows <= 16 && (two || rows > 4) && (long)(N / units + 1) * K * 4 < LDS_PAST && (long)rows * K * 4 < LDS_PAST) {
        const F32Few p{C, A, W, epi, N, K, N / units, N % units};
        auto go = [&](auto kernel, int bytes) {
            if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
            hipLaunchKernelGGL(kernel, dim3(units), dim3(512), bytes, s, F32FewJob<1>{{p}}, rows, 0);
            return true;
        };
        if (two ? go(gemm_f32_few_ring_kernel<2, 2, 1>, FewRing<2, 2>::LDS) : go(gemm_f32_few_ring_kernel<1, 2, 1>, FewRing<1, 2>::LDS)) return;
    }
#define FEW(CT, RT, D) hipLaunchKernelGGL((gemm_f32_few_kernel<CT, RT, D, ROWS>), dim3(groups), dim3(512), 0, s, C, A, W, epi, M, N, K)
    for (int at = 0; at < rows; at += 64) {  // more than 64 rows: where tiles cannot address K
        const int M = rows - at < 64 ? rows - at : 64;
        if (M <= 16) { if (two) FEW(1, 2, 2); else FEW(1, 1, 2); }
        else if (M <= 32) { if (two) FEW(2, 2, 2); else FEW(2, 1, 2); }
        else { if (two) FEW(4, 2, 1); else FEW(4, 1, 1); }
        A += 64L * K, C += 64L * N;
        if (epi.add1) epi.add1 += 64L * N;
        if (epi.add2) epi.add2 += 64L * N;
    }
#undef FEW
}

template <int FP, int FQ, int ROWS>
static int launch_tiles(const F32Tiles& job, const F32Epilogue& epi, hipStream_t s) {
    const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_f32_tile_kernel<FP, FQ, ROWS>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes(FP, FQ));
    PTA_REQUIRE(raised == hipSuccess, "gemm_f32: %d bytes of LDS were refused", lds_bytes(FP, FQ));
    const int R = job.tiles_p * job.tiles_q - job.whole;
    const int groups = (job.whole + 7) / 8 * 8 + (R * job.share + 7) / 8 * 8;
    hipLaunchKernelGGL((gemm_f32_tile_kernel<FP, FQ, ROWS>), dim3(groups), dim3(512), lds_bytes(FP, FQ), s, job, epi);
    if (R > 0) hipLaunchKernelGGL((gemm_f32_add_kernel<FP, FQ, ROWS>), dim3(R * 2 * FP * FQ), dim3(256), 0, s, job, epi);
    return pta_check_launch("gemm_f32");
}

template <int ROWS>
static int launch_plan(const F32Plan& p, const F32Tiles& job, const F32Epilogue& epi, hipStream_t s) {
    if (p.fp == 0) {
        launch_few<ROWS>(job.C, job.A, job.W, epi, job.M, job.N, job.K, s);
        return pta_check_launch("gemm_f32");
    }
    switch (p.fp * 8 + p.fq) {
        case 17: return launch_tiles<2, 1, ROWS>(job, epi, s);
        case 18: return launch_tiles<2, 2, ROWS>(job, epi, s);
        case 19: return launch_tiles<2, 3, ROWS>(job, epi, s);
        case 20: return launch_tiles<2, 4, ROWS>(job, epi, s);
        case 33: return launch_tiles<4, 1, ROWS>(job, epi, s);
        case 34: return launch_tiles<4, 2, ROWS>(job, epi, s);
        case 35: return launch_tiles<4, 3, ROWS>(job, epi, s);
        default: return launch_tiles<4, 4, ROWS>(job, epi, s);
    }
}

static long scratch_values(const F32Plan& p, int M, int N, int K) {
    if (p.fp == 0) return 0;
    const long tiles = (long)((N + 64 * p.fp - 1) / (64 * p.fp)) * ((M + 32 * p.fq - 1) / (32 * p.fq));
    return (tiles - p.whole) * segments(K) * p.fp * p.fq * 2048;
}

// 32-bit values of scratch memory that pta_gemm_f32 needs for this product (0: none)
extern "C" long pta_gemm_f32_scratch(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    return scratch_values(f32_plan(M, N, K), M, N, K);
}

static int f32_run(F32Plan p, float* C, const float* A, const float* W, const float* bias, const float* add1,
                   const float* add2, int M, int N, int K, int act, float* scratch, void* stream) {
    PTA_REQUIRE(C && A && W, "gemm_f32: null pointer");
    PTA_REQUIRE(pta_act_known(act), "gemm_f32: unknown activation %d", act);
    PTA_REQUIRE(scratch_values(p, M, N, K) == 0 || scratch, "gemm_f32: this product needs scratch memory (pta_gemm_f32_scratch)");
    bool wide = N % 4 == 0;
    for (const void* q : {(const void*)C, (const void*)add1, (const void*)add2, (const void*)scratch}) wide = wide && (uintptr_t)q % 16 == 0;
    const F32Epilogue epi{bias, add1, add2, act, wide};
    F32Tiles job{C, scratch, A, W, M, N, K, 0, 0, p.whole, p.share};
    if (p.fp) {
        job.tiles_q = (M + 32 * p.fq - 1) / (32 * p.fq);
        job.tiles_p = (N + 64 * p.fp - 1) / (64 * p.fp);
    }
    const bool vec = K % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
    hipStream_t s = (hipStream_t)stream;
    if (vec && K % BK == 0) return launch_plan<ROW_WHOLE>(p, job, epi, s);
    if (vec) return launch_plan<ROW_VECTORS>(p, job, epi, s);
    return launch_plan<ROW_ELEMENTS>(p, job, epi, s);
}

extern "C" int pta_gemm_f32(float* C, const float* A, const float* W, const float* bias, const float* add1,
                            const float* add2, int M, int N, int K, int act, float* scratch, void* stream) {
    PTA_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: sizes must be positive (M=%d N=%d K=%d)", M, N, K);
    PTA_REQUIRE(M <= 65535 * 64, "gemm_f32: M=%d is too large for one launch", M);
    return f32_run(f32_plan(M, N, K), C, A, W, bias, add1, add2, M, N, K, act, scratch, stream);
}

// How two products of up to sixteen rows run in one launch, or none (units 0) where they do not: each of them one that the kernels for
// few rows have, rows sixteen-byte aligned, 32-bit offsets within a workgroup's rows, and the first's results in what LDS is left.
struct F32PairPlan {
    int units, tiles;  // workgroups, and tiles of sixteen rows of W that their rings hold
    int lds;
};

static F32PairPlan f32_pair_plan(int M, int N1, int K1, int N2, int K2, bool add_first) {
    const F32PairPlan none{0, 0, 0};
    if (M < 1 || M > 16 || N1 < 1 || N2 < 1 || K1 < 1 || K2 < 1 || K1 % 4 || K2 % 4 || (add_first && N1 != N2)) return none;
    if (!few_rows(M, N1, K1) || !few_rows(M, N2, K2)) return none;
    const int most = N1 > N2 ? N1 : N2;
    F32PairPlan p;
    p.units = pta_compute_units();
    if (p.units > (most + 3) / 4) p.units = (most + 3) / 4;  // small matrices: four rows a workgroup
    p.tiles = (most + p.units - 1) / p.units > 16 ? 2 : 1;
    const int rings = p.tiles == 2 ? FewRing<2, 2>::LDS : FewRing<1, 2>::LDS;
    const long kept = add_first ? (N1 / p.units + 1) * 64L : 0;
    if (rings + kept > 160 * 1024) return none;
    for (const long bytes : {(N1 / p.units + 1L) * K1 * 4, (N2 / p.units + 1L) * K2 * 4, (long)M * K1 * 4, (long)M * K2 * 4})
        if (bytes >= LDS_PAST) return none;
    p.lds = rings + (int)kept;
    return p;
}

extern "C" int pta_gemm_f32_pair_ok(int M, int N1, int K1, int N2, int K2, int add_first) {
    return f32_pair_plan(M, N1, K1, N2, K2, add_first != 0).units > 0;
}

// C1 = act1(A1 . W1^T + bias1) and C2 = act2(A2 . W2^T + bias2), or with C1 null the one result C2 = act2(A2 . W2^T + bias2) +
// act1(A1 . W1^T + bias1) + add, from one launch: the values that pta_gemm_f32 gives, bit by bit.
extern "C" int pta_gemm_f32_pair(float* C1, const float* A1, const float* W1, const float* bias1, int N1, int K1, int act1,
                                 float* C2, const float* A2, const float* W2, const float* bias2, int N2, int K2, int act2,
                                 const float* add, int M, void* stream) {
    PTA_REQUIRE(A1 && W1 && C2 && A2 && W2, "gemm_f32_pair: null pointer");
    PTA_REQUIRE(pta_act_known(act1) && pta_act_known(act2), "gemm_f32_pair: unknown activation %d or %d", act1, act2);
    PTA_REQUIRE(!C1 || !add, "gemm_f32_pair: an addition goes with the sum of the two");
    for (const void* q : {(const void*)A1, (const void*)W1, (const void*)A2, (const void*)W2})
        PTA_REQUIRE((uintptr_t)q % 16 == 0, "gemm_f32_pair: rows must be 16-byte aligned");
    const F32PairPlan p = f32_pair_plan(M, N1, K1, N2, K2, !C1);
    PTA_REQUIRE(p.units > 0, "gemm_f32_pair: no launch for %d rows by %d x %d and %d x %d", M, N1, K1, N2, K2);
    const F32Few a{C1, A1, W1, F32Epilogue{bias1, nullptr, nullptr, act1, 0}, N1, K1, N1 / p.units, N1 % p.units};
    const F32Few b{C2, A2, W2, F32Epilogue{bias2, add, nullptr, act2, 0}, N2, K2, N2 / p.units, N2 % p.units};
    auto kernel = p.tiles == 2 ? gemm_f32_few_ring_kernel<2, 2, 2> : gemm_f32_few_ring_kernel<1, 2, 2>;
    PTA_REQUIRE(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, p.lds) == hipSuccess,
                "gemm_f32_pair: %d bytes of LDS were refused", p.lds);
    hipLaunchKernelGGL(kernel, dim3(p.units), dim3(512), p.lds, (hipStream_t)stream, F32FewJob<2>{{a, b}}, M, C1 ? 0 : 1);
    return pta_check_launch("gemm_f32_pair");
}

// pta_gemm_f32 with the choice in the caller's hands, for measuring one against another and for tests of each: fp = 0 for the
// kernel for few rows, else fp 2 or 4 and fq 1 to 4; `room` 32-bit values at scratch.
extern "C" int pta_gemm_f32_as(float* C, const float* A, const float* W, const float* bias, const float* add1,
                               const float* add2, int M, int N, int K, int act, int fp, int fq, int whole, int share,
                               float* scratch, long room, void* stream) {
    PTA_REQUIRE(M > 0 && N > 0 && K > 0 && M <= 65535 * 64, "gemm_f32: sizes out of range (M=%d N=%d K=%d)", M, N, K);
    PTA_REQUIRE(fp == 0 || ((fp == 2 || fp == 4) && fq >= 1 && fq <= 4), "gemm_f32: no tiles of 64 x %d by 32 x %d", fp, fq);
    const F32Plan p{fp, fq, whole, share, 0.0};
    if (fp) {
        const long tiles = (long)((N + 64 * fp - 1) / (64 * fp)) * ((M + 32 * fq - 1) / (32 * fq));
        PTA_REQUIRE(K <= MOST_K && whole >= 0 && whole <= tiles && share >= 1 && share <= segments(K),
                    "gemm_f32: %d of %ld tiles whole, %d shares of %d segments", whole, tiles, share, segments(K));
    }
    PTA_REQUIRE(scratch_values(p, M, N, K) <= room, "gemm_f32: room for %ld sums, %ld are needed", room, scratch_values(p, M, N, K));
    return f32_run(p, C, A, W, bias, add1, add2, M, N, K, act, scratch, stream);
}
