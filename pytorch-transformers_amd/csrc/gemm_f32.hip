// C[M,N] = act(A[M,K] . W[N,K]^T + bias) + add1 + add2 in true 32-bit, on the 32-bit matrix instruction
// (v_mfma_f32_16x16x4_f32: products and sums in 32-bit, 154 TFLOP/s dense on this chip; the vector units give half).
// The 32-bit path of the whole model runs its projections, feed-forwards and output head through here.
//
// Order of summation.  A row's result is bitwise the same alone and in any batch, so every kernel here sums the products
// of an output in one order, which K alone decides: K is walked in blocks of sixteen elements (the last one filled up with
// zeros), the blocks are cut into up to eight segments of equal length, a segment is one chain of matrix instructions
// (a block is four instructions; each takes one element in four, from 3, 7, 11 and 15 down to 0, 4, 8 and 12, so that a
// lane's four operands are sixteen consecutive bytes of a row), and the segments' sums are added in order.  Where a row lies in
// the grid, which kernel runs and how many workgroups share the segments changes nothing.
//
// The error against 64 bits, relative to the root of the sum of a row's squared products, is 3.7 x 2^-24 at K = 1,040, 7.2 at
// 4,544 and 14.3 at 18,176 (rms).  Whether a block's four instructions go down or up makes no difference to it (7.22 and 7.21 at
// 4,544, 14.31 and 14.31 at 18,176; down was the smaller in 56 of 144 draws): down is what it is, and every kernel has to keep to it.
//
// Measured at 4,544 / 18,176 features (one kernel of 64 x 64 tiles on the vector units before): one row of A 986 -> 56 us a
// product on average (22 us = 3.7 TB/s for 83 MB, 70 to 75 us = 4.4 to 4.7 TB/s for 330 MB); 2,053 rows 26 -> 103 to 131 TFLOP/s.
//
// Three ways to the same numbers, by what bounds them:
//   few rows (M <= 32, with a short K 64): every weight is read once and that is the time.  A workgroup owns up to 32 rows of W and its eight
//     waves a segment each; W goes from memory straight into the instruction's operands, the sums meet in LDS.
//   many rows: tiles of 128 x 128 or 64 x 64 through two LDS buffers, bound by the matrix instruction (loads straight to LDS
//     where rows are sixteen-byte aligned, else through registers).
//   in between, or N small: too few tiles to fill the chip, so the segments of a tile are shared out over workgroups, whose
//     sums go to memory and are added by a small launch.
#include "common.h"
#include "pta_kernels.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define SEGS 8          // segments of K, at most
#define SKINNY_ROWS 32  // rows of A up to which the kernel for few rows runs
#define SHARE_K 1024    // K from which segments may be shared out over workgroups

struct F32Epilogue {
    const float* bias;
    const float* add1;
    const float* add2;
    int act;
};

__device__ __forceinline__ float finish(float v, const F32Epilogue& e, int n, long at) {
    if (e.bias) v += e.bias[n];
    if (e.act) v = apply_act(v, e.act);
    if (e.add1) v += e.add1[at];
    if (e.add2) v += e.add2[at];
    return v;
}

// How rows are read: element by element; sixteen bytes at a time (rows sixteen-byte aligned, K a multiple of 4); the same
// without a look at the end (K a multiple of 16, what every published size is).
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

__host__ __device__ static inline int seg_blocks(int K) { return ((K + 15) / 16 + SEGS - 1) / SEGS; }

// ---- few rows ---------------------------------------------------------------------------------------------------------
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
    const int nb = (K + 15) / 16, sb = seg_blocks(K);
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

    f32x4 w[2][D][RT], x[2][D][CT];
    auto fetch = [&](int buf, int b) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            const int k = 16 * min(b + i, b1 - 1) + kq;  // past the segment: its last block again, not used
#pragma unroll
            for (int r = 0; r < RT; ++r) w[buf][i][r] = load4<ROWS>(wr[r], k, K);
#pragma unroll
            for (int c = 0; c < CT; ++c) x[buf][i][c] = load4<ROWS>(xr[c], k, K);
        }
    };
    auto multiply = [&](int buf, int b) {
#pragma unroll
        for (int i = 0; i < D; ++i) {
            if (b + i < b1) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int r = 0; r < RT; ++r)
#pragma unroll
                        for (int c = 0; c < CT; ++c)
                            acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[buf][i][r][3 - j], x[buf][i][c][3 - j], acc[r][c], 0, 0, 0);
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
        const int t = i >> 6, l = i & 63;
        f32x4 v = part[0][t][l];
        for (int s = 1; s < used; ++s) {
            const f32x4 p = part[s][t][l];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] += p[j];
        }
        const int m = 16 * (t % CT) + (l & 15);
        const int n = n0 + 16 * (t / CT) + 4 * (l >> 4);
        if (m < M) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (n + j < n1) C[(long)m * N + n + j] = finish(v[j], epi, n + j, (long)m * N + n + j);
        }
    }
}

// ---- many rows ----------------------------------------------------------------------------------------------------------
// A workgroup of four waves, two by two, on a tile of T x T.  A row of a tile is 32 elements of K in LDS, 36 apart: the eight
// lanes that read together (rows next to each other, sixteen bytes each) then cover every bank once.
#define BK 32
#define PITCH 36

template <int T, bool SPLIT>
__global__ __launch_bounds__(256, 2) void gemm_f32_tile_kernel(float* __restrict__ C, const float* __restrict__ A,
                                                               const float* __restrict__ W, F32Epilogue epi, int M, int N,
                                                               int K, int tiles_m, int tiles_n) {
    constexpr int F = T / 32;        // tiles of sixteen rows per wave and side
    constexpr int L = T * 8 / 256;   // sixteen-byte loads per thread and side
    __shared__ float As[2][T * PITCH];
    __shared__ float Ws[2][T * PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, kq = 4 * (lane >> 4);
    // workgroups go to the eight dies in turn: give each die a run of tiles that share rows of W, which its L2 then holds
    const int tiles = tiles_m * tiles_n;
    const int per = (tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || tile >= tiles) return;
    const int m0 = (tile % tiles_m) * T, n0 = (tile / tiles_m) * T;
    const int wn = (wave & 1) * (T / 2), wm = (wave >> 1) * (T / 2);
    const int nb = (K + 15) / 16, sb = seg_blocks(K);
    // SPLIT: this workgroup's share of the segments
    const int used = (nb + sb - 1) / sb;
    const int s0 = SPLIT ? (int)((long)blockIdx.y * used / gridDim.y) : 0;
    const int s1 = SPLIT ? (int)((long)(blockIdx.y + 1) * used / gridDim.y) : used;
    const int b_first = s0 * sb, b_last = min(nb, s1 * sb);

    f32x4 acc[F][F], total[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 ra[L], rw[L];
    const float* pa[L];
    const float* pw[L];
#pragma unroll
    for (int i = 0; i < L; ++i) {
        const int row = (tid + 256 * i) >> 3;
        pa[i] = A + (long)min(m0 + row, M - 1) * K;
        pw[i] = W + (long)min(n0 + row, N - 1) * K;
    }
    const int kc = 4 * (tid & 7);
    auto fetch = [&](int b) {  // blocks b and b + 1
        const int k = 16 * b + kc;
#pragma unroll
        for (int i = 0; i < L; ++i) {
            ra[i] = load4<ROW_ELEMENTS>(pa[i], k, K);
            rw[i] = load4<ROW_ELEMENTS>(pw[i], k, K);
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int at = ((tid + 256 * i) >> 3) * PITCH + kc;
            *(f32x4*)&As[buf][at] = ra[i];
            *(f32x4*)&Ws[buf][at] = rw[i];
        }
    };
    auto store_all = [&](const f32x4 (&v)[F][F], float* to, bool last) {
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j) {
                const int n = n0 + wn + 16 * i + kq, m = m0 + wm + 16 * j + r16;
                if (m >= M) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) to[(long)m * N + n + e] = last ? finish(v[i][j][e], epi, n + e, (long)m * N + n + e) : v[i][j][e];
            }
    };
    if (b_first < b_last) {
        fetch(b_first);
        stage(0);
        __syncthreads();
    }
    int left = sb, segs = 0, buf = 0;  // blocks left of the segment, segments finished
    for (int b = b_first; b < b_last; b += 2, buf ^= 1) {
        const bool more = b + 2 < b_last;
        if (more) fetch(b + 2);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (b + h < b_last) {
                f32x4 w[F], x[F];
#pragma unroll
                for (int i = 0; i < F; ++i) {
                    w[i] = *(const f32x4*)&Ws[buf][(wn + 16 * i + r16) * PITCH + 16 * h + kq];
                    x[i] = *(const f32x4*)&As[buf][(wm + 16 * i + r16) * PITCH + 16 * h + kq];
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int i = 0; i < F; ++i)
#pragma unroll
                        for (int c = 0; c < F; ++c)
                            acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[i][3 - j], x[c][3 - j], acc[i][c], 0, 0, 0);
                if (--left == 0 || b + h + 1 == b_last) {  // the segment ends: its sum joins the others in their order
                    if (SPLIT) {
                        store_all(acc, C + (long)(s0 + segs) * M * N, false);
                    } else if (segs == 0) {
#pragma unroll
                        for (int i = 0; i < F; ++i)
#pragma unroll
                            for (int c = 0; c < F; ++c) total[i][c] = acc[i][c];
                    } else {
#pragma unroll
                        for (int i = 0; i < F; ++i)
#pragma unroll
                            for (int c = 0; c < F; ++c)
#pragma unroll
                                for (int e = 0; e < 4; ++e) total[i][c][e] += acc[i][c][e];
                    }
#pragma unroll
                    for (int i = 0; i < F; ++i)
#pragma unroll
                        for (int c = 0; c < F; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
                    ++segs;
                    left = sb;
                }
            }
        }
        if (more) {
            stage(buf ^ 1);  // the other buffer: everyone is past reading it since the last barrier
            __syncthreads();
        }
    }
    if (!SPLIT) store_all(total, C, true);
}

// The same tiles where rows can be read sixteen bytes at a time (rows sixteen-byte aligned, K a multiple of 4), loads going
// straight to LDS.  A row of a tile is 32 elements of K, 128 bytes without a gap: sixteen bytes c of row r lie at place
// c ^ (r % 8), so that the eight lanes that read together cover every bank once.
//
// What bounds it is the matrix instruction (32 cycles each); the kernel above, which stages through registers and reads a
// block's operands right before their products, keeps it busy 80 % of the time a workgroup is there.  Here operands of a
// block are read while the block before is multiplied, and the loads of a step have the whole step before it to arrive:
// 8,192 x 8,192 x 4,096 124 -> 139 TFLOP/s, 2,053 rows by 4,544 x 4,544 90 -> 113, by 18,176 x 4,544 110 -> 131.
// TAIL: K is no multiple of 16, what a block holds past it has to be zero.

// sixteen bytes a lane from byte `at` of an array of `bytes` into LDS, one lane after the other; zeros from its end on
__device__ __forceinline__ void to_lds(const float* src, int bytes, float* dst, int at) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, bytes, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, at, 0, 0, 0);
}

template <int T, bool TAIL, bool SPLIT>
__global__ __launch_bounds__(256, 2) void gemm_f32_stream_kernel(float* __restrict__ C, const float* __restrict__ A,
                                                                 const float* __restrict__ W, F32Epilogue epi, int M, int N,
                                                                 int K, int tiles_m, int tiles_n) {
    constexpr int F = T / 32;       // tiles of sixteen rows per wave and side
    constexpr int L = T * 8 / 256;  // sixteen-byte loads per thread and side
    // A's rows, then W's; two arrays, so that the compiler sees which of them a load is on its way to
    __shared__ __attribute__((aligned(1024))) float lds0[2 * T * BK];
    __shared__ __attribute__((aligned(1024))) float lds1[2 * T * BK];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, kq = 4 * (lane >> 4);
    const int tiles = tiles_m * tiles_n;
    const int per = (tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || tile >= tiles) return;
    const int m0 = (tile % tiles_m) * T, n0 = (tile / tiles_m) * T;
    const int wn = (wave & 1) * (T / 2), wm = (wave >> 1) * (T / 2);
    const int nb = (K + 15) / 16, sb = seg_blocks(K);
    const int used = (nb + sb - 1) / sb;
    const int s0 = SPLIT ? (int)((long)blockIdx.y * used / gridDim.y) : 0;
    const int s1 = SPLIT ? (int)((long)(blockIdx.y + 1) * used / gridDim.y) : used;
    const int b_first = s0 * sb, b_last = min(nb, s1 * sb);

    f32x4 acc[F][F], total[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const float* at_a = A + (long)m0 * K;
    const float* at_w = W + (long)n0 * K;
    const int bytes_a = min(T, M - m0) * K * 4, bytes_w = min(T, N - n0) * K * 4;
    const int trow = tid >> 3, kc = 4 * ((tid & 7) ^ (trow & 7));
    // blocks b and b + 1; rows past the last are zeros, what the second block holds past K is not used; past b_last nothing is read
    auto fetch = [&](float* buf, int b) __attribute__((always_inline)) {
        const int k = 16 * b + kc;
#pragma unroll
        for (int i = 0; i < L; ++i) {
            const int at = TAIL && k >= K ? -16 : ((trow + 32 * i) * K + k) * 4;
            to_lds(at_a, b < b_last ? bytes_a : 0, buf + (32 * i + 8 * wave) * BK, at);
            to_lds(at_w, b < b_last ? bytes_w : 0, buf + (T + 32 * i + 8 * wave) * BK, at);
        }
    };
    f32x4 w[2][F], x[2][F];
    const int place[2] = {4 * ((lane >> 4) ^ (r16 & 7)), 4 * ((4 + (lane >> 4)) ^ (r16 & 7))};
    auto read = [&](const float* buf, int h) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < F; ++i) {
            x[h][i] = *(const f32x4*)&buf[(wm + 16 * i + r16) * BK + place[h]];
            w[h][i] = *(const f32x4*)&buf[(T + wn + 16 * i + r16) * BK + place[h]];
        }
    };
    auto store_all = [&](const f32x4 (&v)[F][F], float* to, bool last) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j) {
                const int n = n0 + wn + 16 * i + kq, m = m0 + wm + 16 * j + r16;
                if (m >= M) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) to[(long)m * N + n + e] = last ? finish(v[i][j][e], epi, n + e, (long)m * N + n + e) : v[i][j][e];
            }
    };
    int left = sb, segs = 0;  // blocks left of the segment, segments finished
    auto multiply = [&](int h, int b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int c = 0; c < F; ++c)
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[h][i][3 - j], x[h][c][3 - j], acc[i][c], 0, 0, 0);
        if (--left == 0 || b + 1 == b_last) {  // the segment ends: its sum joins the others in their order
            if (SPLIT) {
                store_all(acc, C + (long)(s0 + segs) * M * N, false);
            } else {
                const bool first = segs == 0;
#pragma unroll
                for (int i = 0; i < F; ++i)
#pragma unroll
                    for (int c = 0; c < F; ++c)
#pragma unroll
                        for (int e = 0; e < 4; ++e) total[i][c][e] = first ? acc[i][c][e] : total[i][c][e] + acc[i][c][e];
            }
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int c = 0; c < F; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};
            ++segs;
            left = sb;
        }
    };
    // Blocks b and b + 1 out of `cur`.  Everyone has read all of it when its second block is multiplied: then it takes the loads
    // of the step after next, and the next step's first block is read.
    auto step = [&](float* cur, const float* next, int b) __attribute__((always_inline)) {
        read(cur, 1);
        __builtin_amdgcn_sched_barrier(0);
        if (b < b_last) multiply(0, b);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070);  // this wave's reads of `cur` are done, its loads into `next` have landed
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        fetch(cur, b + 4);
        read(next, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (b + 1 < b_last) multiply(1, b + 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (b_first < b_last) {
        fetch(lds0, b_first);
        fetch(lds1, b_first + 2);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read(lds0, 0);
        for (int b = b_first; b < b_last; b += 4) {
            step(lds0, lds1, b);
            step(lds1, lds0, b + 2);
        }
        __builtin_amdgcn_s_waitcnt(0x0070);  // nothing is on its way to LDS when the workgroup ends
    }
    if (!SPLIT) store_all(total, C, true);
}

// the segments' sums added in order, and the epilogue
__global__ void gemm_f32_add_kernel(float* __restrict__ C, const float* __restrict__ part, F32Epilogue epi, int segs, long MN, int N) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= MN) return;
    float v = part[i];
    for (int s = 1; s < segs; ++s) v += part[(long)s * MN + i];
    C[i] = finish(v, epi, (int)(i % N), i);
}

// How a product runs: the tile's side (0: the kernel for few rows) and over how many workgroups a tile's segments are shared.
static void f32_plan(int M, int N, int K, int* tile, int* share) {
    *tile = 0, *share = 1;
    // 33 rows by 4,544 x 4,544: 61 us with the kernel for few rows, 36 with shared tiles; 17 rows: 35 and 51; 33 rows by 256 x
    // 512, whose segments are too short to be shared: 7 and 13
    if (M <= (K < SHARE_K ? 2 * SKINNY_ROWS : SKINNY_ROWS)) return;
    const int cus = 256;
    auto tiles = [&](long t) { return ((M + t - 1) / t) * ((N + t - 1) / t); };
    auto rounds = [&](long n) { return (double)((n + cus - 1) / cus); };
    // time of a round: a tile of 128 is four of 64, which read twice as much per product (8,192 x 8,192 x 4,096: 139 and
    // 134 TFLOP/s; 2,053 x 4,544 x 4,544, where 128 leaves the last round half empty: 101 and 119)
    const double big = 4.0 * rounds(tiles(128)), small = 1.04 * rounds(tiles(64));
    *tile = big <= small ? 128 : 64;
    const int used = ((K + 15) / 16 + seg_blocks(K) - 1) / seg_blocks(K);
    if (*tile == 64 && K >= SHARE_K)  // a chip that is not filled twice: share the segments out
        while (*share < used && tiles(64) * *share < 2 * cus) *share *= 2;
    if (*share > used) *share = used;
}

// 32-bit values of scratch memory that pta_gemm_f32 needs for this product (0: none)
extern "C" long pta_gemm_f32_scratch(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    int tile, share;
    f32_plan(M, N, K, &tile, &share);
    if (share <= 1) return 0;
    return (long)(((K + 15) / 16 + seg_blocks(K) - 1) / seg_blocks(K)) * M * N;
}

template <int ROWS>
static void launch_few(float* C, const float* A, const float* W, const F32Epilogue& epi, int M, int N, int K, hipStream_t s) {
    // whole rounds of the 256 compute units, up to 32 rows of W each; small matrices: four rows a workgroup
    int groups = 256 * ((N + 256 * 32 - 1) / (256 * 32));
    if (groups > (N + 3) / 4) groups = (N + 3) / 4;
    const bool two = (N + groups - 1) / groups > 16;
#define FEW(CT, RT, D) hipLaunchKernelGGL((gemm_f32_few_kernel<CT, RT, D, ROWS>), dim3(groups), dim3(512), 0, s, C, A, W, epi, M, N, K)
    if (M <= 16) { if (two) FEW(1, 2, 4); else FEW(1, 1, 4); }
    else if (M <= 32) { if (two) FEW(2, 2, 4); else FEW(2, 1, 4); }
    else { if (two) FEW(4, 2, 2); else FEW(4, 1, 2); }
#undef FEW
}

static void launch_tiles(float* C, float* scratch, const float* A, const float* W, const F32Epilogue& epi, int M, int N, int K,
                         int tile, int share, bool vec, hipStream_t s) {
    const int tm = (M + tile - 1) / tile, tn = (N + tile - 1) / tile;
    const int groups = 8 * ((tm * tn + 7) / 8);
    // offsets within a tile's rows are 32-bit bytes
    const bool stream = vec && (long)(128 + 2) * K * 4 < (1L << 31);
#define LAUNCH(KERNEL, SPLIT, OUT) \
    hipLaunchKernelGGL(KERNEL, dim3(groups, SPLIT ? share : 1), dim3(256), 0, s, OUT, A, W, epi, M, N, K, tm, tn)
#define TILE(T, SPLIT, OUT) \
    do { \
        if (!stream) LAUNCH((gemm_f32_tile_kernel<T, SPLIT>), SPLIT, OUT); \
        else if (K % 16) LAUNCH((gemm_f32_stream_kernel<T, true, SPLIT>), SPLIT, OUT); \
        else LAUNCH((gemm_f32_stream_kernel<T, false, SPLIT>), SPLIT, OUT); \
    } while (0)
    if (share > 1) TILE(64, true, scratch);
    else if (tile == 128) TILE(128, false, C);
    else TILE(64, false, C);
#undef TILE
#undef LAUNCH
    if (share > 1) {
        const long mn = (long)M * N;
        const int segs = ((K + 15) / 16 + seg_blocks(K) - 1) / seg_blocks(K);
        hipLaunchKernelGGL(gemm_f32_add_kernel, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, s, C, scratch, epi, segs, mn, N);
    }
}

extern "C" int pta_gemm_f32(float* C, const float* A, const float* W, const float* bias, const float* add1,
                            const float* add2, int M, int N, int K, int act, float* scratch, void* stream) {
    PTA_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_f32: sizes must be positive (M=%d N=%d K=%d)", M, N, K);
    PTA_REQUIRE(C && A && W, "gemm_f32: null pointer");
    PTA_REQUIRE(pta_act_known(act), "gemm_f32: unknown activation %d", act);
    PTA_REQUIRE(M <= 65535 * 64, "gemm_f32: M=%d is too large for one launch", M);
    int tile, share;
    f32_plan(M, N, K, &tile, &share);
    PTA_REQUIRE(share <= 1 || scratch, "gemm_f32: this product needs scratch memory (pta_gemm_f32_scratch)");
    const F32Epilogue epi{bias, add1, add2, act};
    const bool vec = K % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
    hipStream_t s = (hipStream_t)stream;
#define BY_ROWS(FN, ...) (vec && K % 16 == 0 ? FN<ROW_WHOLE>(__VA_ARGS__) : vec ? FN<ROW_VECTORS>(__VA_ARGS__) : FN<ROW_ELEMENTS>(__VA_ARGS__))
    if (tile == 0) BY_ROWS(launch_few, C, A, W, epi, M, N, K, s);
    else launch_tiles(C, scratch, A, W, epi, M, N, K, tile, share, vec, s);
#undef BY_ROWS
    return pta_check_launch("gemm_f32");
}
