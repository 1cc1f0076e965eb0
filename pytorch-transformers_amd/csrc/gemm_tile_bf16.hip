// Products of many rows in bfloat16: y[M, N] = act(x[M, K] . W[N, K]^T + bias) + add1 + add2, 32-bit sums.
//
// A workgroup of eight waves (four along the rows of W, two along the rows of x) makes a tile of 256 rows of W by 32 FQ rows of
// x, a block of 64 elements of K at a time.  A wave's 64 x 16 FQ sums stay in its registers; its operands come from LDS,
// the 32 elements of K that are multiplied next being read while the 32 before them are multiplied (two sets of fragments),
// so that the matrix cores wait for LDS only behind the one barrier of a block.  Blocks are fetched straight to LDS, without
// a detour over registers: W, which mostly comes from far away, into three stages, x into two (three where they fit).
//
//   block b:  first set x second set being read, W of block b + 2 asked for
//             wait: the wave's reads of block b are done, its share of block b + 1 has landed; barrier
//             second set x next block's first set being read, x of block b + 2 (b + 3) asked for, into the stage just freed
//
// A row of a stage is 64 elements, 128 bytes without a gap: sixteen bytes c of row r lie at place c ^ (r / 2 % 8), so that
// any sixteen lanes that read together cover every bank once (no conflict in the counters).  The order within a row is made
// on the way in: each lane of a load asks for the sixteen bytes that its place in LDS is to hold.
//
// What bounds it: at 8,192 x 8,192 x 8,192 the matrix cores' power (they run at 1.78 GHz and are busy 77 % of the
// cycles), at fewer rows how many tiles there are for 256 compute units, which is what FQ and the ranges of K are chosen by
// (tile_plan below), and the traffic out of L2, some 25 bytes a cycle and compute unit.
//
// Measured, TFLOP/s of this kernel and of the vendor library's product (M x N x K):
//   2,048 x 18,176 x 4,544  1,264 / 1,097     2,317 x 18,176 x 4,544  1,260 / 916     672 x 4,544 x 18,176  1,058 / 524
//   2,048 x 4,544 x 4,544   1,171 / 1,083     4,740 x 8,192 x 32,768  1,392 / 1,195   895 x 4,160 x 1,040   461 / 332
//   2,583 x 8,192 x 2,048   1,075 / 895       8,192 x 8,192 x 8,192   1,486 / 1,608   25,148 x 16,384 x 4,096 1,368 / 1,452
// Eight waves that take turns, four reading while four multiply, gave the same at FQ = 8 and 5 to 20 % less below; four waves
// with tiles of 128 x 128 need more registers than the compiler places without copies.
#include "common.h"
#include "pta_kernels.h"

#include <type_traits>

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

#define TILE_N 256           // rows of W of a tile
#define TILE_GROUP 8         // tiles along x that stand side by side in the order of tiles
#define TILE_P_STAGES 3
#define TILE_P_BYTES 32768   // a stage of W
#define TILE_LDS_Q (TILE_P_STAGES * TILE_P_BYTES)
#define TILE_PAST 0x7ffffff0  // an offset past the end of every operand: such loads give zeros
#define TILE_PITCH 144        // bytes from row to row of a wave's results on their way out

struct TileJob {
    bf16_t* y;
    float* part;  // sums of the tiles whose K is cut: [range][tile][wave][fragment][lane][4]
    const bf16_t* x;
    const bf16_t* W;
    const float* bias;
    const bf16_t* add1;
    const bf16_t* add2;
    int M, N, K, ldx, ldy;
    int tiles_q, tiles_p;  // tiles along the rows of x and of W
    int whole;             // the first tiles, computed over all of K
    int split;             // ranges of K of the others
};

static constexpr __host__ __device__ int q_stages(int FQ) { return FQ <= 5 ? 3 : 2; }
static constexpr __host__ __device__ int lds_bytes(int FQ) { return TILE_LDS_Q + q_stages(FQ) * FQ * 4096; }

// waits until at most N of the wave's loads are on their way
template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

__device__ __forceinline__ void wait_reads() { __builtin_amdgcn_s_waitcnt(0xc07f); }  // lgkmcnt(0)

__device__ __forceinline__ void meet() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Sixteen bytes a lane from byte `at` of a buffer straight to LDS, one lane after the other from `to` on; zeros past the
// buffer's end.  Written out because the compiler would wait for every such load before any read of LDS; the waits are
// this kernel's own (wait_loads).  There is no register that the load writes.
__device__ __forceinline__ void fetch16(i32x4_t buffer, unsigned to, int at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(at), "s"(buffer) : "memory");
}

__device__ __forceinline__ i32x4_t buffer_of(const void* p, int bytes) {
    const uint64_t at = (uint64_t)(uintptr_t)p;
    return i32x4_t{__builtin_amdgcn_readfirstlane((int)(uint32_t)at), __builtin_amdgcn_readfirstlane((int)((uint32_t)(at >> 32) & 0xffffu)),
                   __builtin_amdgcn_readfirstlane(bytes), 0x00020000};
}

// Tile t: runs of TILE_GROUP tiles along x for one tile of W after the other, so that the tiles that a die works on at a time
// (32 neighbours) share eight blocks of x and four of W, which its L2 then holds.
__device__ __forceinline__ void tile_at(const TileJob& job, int t, int& tp, int& tq) {
    const int per_group = TILE_GROUP * job.tiles_p;
    const int grp = t / per_group, in = t - grp * per_group;
    const int width = min(TILE_GROUP, job.tiles_q - grp * TILE_GROUP);
    tp = in / width;
    tq = grp * TILE_GROUP + in - tp * width;
}

// what follows the product, on eight neighbours of a row: u holds the products rounded to bfloat16
template <int ACT>
__device__ __forceinline__ void store8(const TileJob& job, int m, int n, uint4 u) {
    if (ACT != PTA_ACT_NONE || job.bias || job.add1 || job.add2) {
        float v[8];
        unpack8(u, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (job.bias) v[e] = round_to_bf16(v[e] + job.bias[n + e]);
            if (ACT != PTA_ACT_NONE) v[e] = apply_act_bf16(v[e], ACT);
        }
        if (job.add1 || job.add2) {
            const uint4 none = make_uint4(0u, 0u, 0u, 0u);
            const uint4 u1 = job.add1 ? *reinterpret_cast<const uint4*>(job.add1 + (long)m * job.N + n) : none;
            const uint4 u2 = job.add2 ? *reinterpret_cast<const uint4*>(job.add2 + (long)m * job.N + n) : none;
            float x1[8], x2[8];
            unpack8(u1, x1);
            unpack8(u2, x2);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] += x1[e];  // an absent addend is zeros: the arithmetic is epilogue_bf16x8_kernel's
                v[e] += x2[e];
            }
        }
        u = pack8(v);
    }
    *reinterpret_cast<uint4*>(job.y + (long)m * job.ldy + n) = u;
}

template <int FQ, int ACT>
__global__ __launch_bounds__(512, 2) void gemm_tile_kernel(TileJob job) {
    constexpr int TILE_M = 32 * FQ, SQ = q_stages(FQ), Q_BYTES = TILE_M * 128, READS = 4 + FQ;
    static_assert(lds_bytes(FQ) <= 160 * 1024 && 8 * FQ * 16 * TILE_PITCH <= lds_bytes(FQ), "the stages and the results must fit LDS");
    extern __shared__ __attribute__((aligned(1024))) char lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wp = wave & 3, wq = wave >> 2;
    const int M = job.M, N = job.N, K = job.K;
    const int tiles = job.tiles_p * job.tiles_q, blocks = (K + 63) >> 6;
    // which tile, which range of K: workgroups go to the eight dies in turn, each die takes a run of tiles
    int t, b0 = 0, b1 = blocks, range = 0, rest = -1;
    const int whole8 = (job.whole + 7) >> 3;
    if ((int)blockIdx.x < whole8 * 8) {
        t = (blockIdx.x & 7) * whole8 + (blockIdx.x >> 3);
        if (t >= job.whole) return;
    } else {
        const int R = tiles - job.whole, all = R * job.split, per = (all + 7) >> 3;
        const int i = blockIdx.x - whole8 * 8, at = (i & 7) * per + (i >> 3);
        if (at >= all) return;
        range = at / R;
        rest = at - range * R;
        t = job.whole + rest;
        b0 = (int)((long)blocks * range / job.split);
        b1 = (int)((long)blocks * (range + 1) / job.split);
    }
    int tp, tq;
    tile_at(job, t, tp, tq);
    const int n0 = tp * TILE_N, m0 = tq * TILE_M;

    // A wave's load fills eight rows.  Rows past the last one lie past the buffer's end; elements past K (or past the
    // range's end, where nothing more is needed) are asked for there.
    const i32x4_t rw = buffer_of(job.W, N * K * 2), rx = buffer_of(job.x, ((M - 1) * job.ldx + K) * 2);
    const int row8 = wave * 8 + (lane >> 3);
    const int c8 = ((lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7)) * 8;  // first element of the lane's chunk within a block
    const int at_w = ((n0 + row8) * K + c8) * 2, at_x = ((m0 + row8) * job.ldx + c8) * 2;
    const int k_end = min(K, b1 * 64);

    f32x4_t acc[4][FQ];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < FQ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    const int r16 = lane & 15, c4 = lane >> 4;
    const int in_row = r16 * 128 + ((c4 ^ (r16 >> 1)) * 16);  // the second 32 elements of K: 64 flipped
    const int ap = wp * 8192 + in_row, aq = TILE_LDS_Q + wq * (FQ * 2048) + in_row;
    const unsigned to = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds + wave * 1024;

    // G: which half of the waves; the 4 FQ loads of a block of x are shared out to eight waves
    auto run = [&](auto group_c) {
        constexpr int G = decltype(group_c)::value;
        constexpr int NQ = (FQ + 1 - G) / 2;
        int kp = b0 * 64, kq = b0 * 64, sp = 0, sq = 0;  // the block that is asked for next, and the stage it goes to
        auto load_w = [&](int l) {
            fetch16(rw, to + sp + l * 8192, kp + c8 < k_end ? at_w + (kp + l * 64 * K) * 2 : TILE_PAST);
            if (l == 3) { kp += 64; sp = sp == (TILE_P_STAGES - 1) * TILE_P_BYTES ? 0 : sp + TILE_P_BYTES; }
        };
        auto load_x = [&](int l) {
            fetch16(rx, to + TILE_LDS_Q + sq + l * 8192, kq + c8 < k_end ? at_x + (kq + l * 64 * job.ldx) * 2 : TILE_PAST);
            if (l == NQ - 1) { kq += 64; sq = sq == (SQ - 1) * Q_BYTES ? 0 : sq + Q_BYTES; }
        };
        auto all_w = [&]() {
#pragma unroll
            for (int l = 0; l < 4; ++l) load_w(l);
        };
        auto all_x = [&]() {
#pragma unroll
            for (int l = 0; l < NQ; ++l) load_x(l);
        };
        bf16x8_t p[2][4], q[2][FQ];
        auto read = [&](int stage_p, int stage_q, int set, int n) {  // the n-th fragment of a set
            if (n < 4) p[set][n] = *reinterpret_cast<const bf16x8_t*>(lds + ((ap ^ (set * 64)) + stage_p) + n * 2048);
            else q[set][n - 4] = *reinterpret_cast<const bf16x8_t*>(lds + ((aq ^ (set * 64)) + stage_q) + (n - 4) * 2048);
        };
        auto multiply = [&](int set, int j) {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(p[set][i], q[set][j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        };
        all_w();
        all_x();
        all_w();
        all_x();
        if (SQ == 3) all_x();
        wait_loads<4 + NQ * (SQ - 1)>();  // the first block's
        meet();
        int cp = 0, cq = 0;
#pragma unroll
        for (int n = 0; n < READS; ++n) read(0, 0, 0, n);
        for (int b = b0; b < b1; ++b) {
            const int np = cp == (TILE_P_STAGES - 1) * TILE_P_BYTES ? 0 : cp + TILE_P_BYTES;
            const int nq = cq == (SQ - 1) * Q_BYTES ? 0 : cq + Q_BYTES;
#pragma unroll
            for (int j = 0; j < FQ; ++j) {
#pragma unroll
                for (int n = 0; n < READS; ++n)
                    if (n / 2 == j || (j == FQ - 1 && n / 2 > j)) read(cp, cq, 1, n);
#pragma unroll
                for (int l = 0; l < 4; ++l)
                    if (l * FQ / 4 == j) load_w(l);
                multiply(0, j);
            }
            wait_reads();
            wait_loads<4 + (SQ == 3 ? NQ : 0)>();  // all but W two blocks on (and x two blocks on)
            meet();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FQ; ++j) {
#pragma unroll
                for (int n = 0; n < READS; ++n)
                    if (n / 2 == j || (j == FQ - 1 && n / 2 > j)) read(np, nq, 0, n);
#pragma unroll
                for (int l = 0; l < NQ; ++l)
                    if (l * FQ / NQ == j) load_x(l);
                multiply(1, j);
            }
            cp = np;
            cq = nq;
        }
        wait_loads<0>();  // nothing is on its way to LDS any more
    };
    if (wq == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});

    if (rest >= 0) {
        f32x4_t* out = reinterpret_cast<f32x4_t*>(job.part) + (((long)range * (tiles - job.whole) + rest) * 8 + wave) * (4 * FQ * 64) + lane;
#pragma unroll
        for (int j = 0; j < FQ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) out[(j * 4 + i) * 64] = acc[i][j];
        return;
    }
    // Through LDS, so that a store takes whole lines, eight rows of 64 columns (each lane's four neighbours straight to memory
    // took 11 us a tile of 256 x 256 where this takes 6).
    meet();  // everyone is past reading the last block
    char* mine = lds + wave * (FQ * 16 * TILE_PITCH);
#pragma unroll
    for (int j = 0; j < FQ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            union { bf16_t h[4]; uint2 u; } o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o.h[e] = f32_to_bf16_bits(acc[i][j][e]);
            *reinterpret_cast<uint2*>(mine + (j * 16 + r16) * TILE_PITCH + (i * 16 + c4 * 4) * 2) = o.u;
        }
    const int n = n0 + wp * 64 + (lane & 7) * 8;
#pragma unroll
    for (int j = 0; j < 2 * FQ; ++j) {
        const int row = j * 8 + (lane >> 3), m = m0 + wq * (FQ * 16) + row;
        const uint4 u = *reinterpret_cast<const uint4*>(mine + row * TILE_PITCH + (lane & 7) * 16);
        if (m < M && n < N) store8<ACT>(job, m, n, u);
    }
}

// The tiles whose K was cut: the ranges' sums added in order, then as above.  A workgroup has the four fragments of sixteen
// rows of x by 64 of W of a wave (a fragment a wave), a lane four neighbours of a row; they change hands through LDS.
template <int FQ, int ACT>
__global__ __launch_bounds__(256) void gemm_tile_reduce_kernel(TileJob job) {
    __shared__ __attribute__((aligned(16))) char rows[16 * TILE_PITCH];
    const int R = job.tiles_p * job.tiles_q - job.whole;
    const int lane = threadIdx.x & 63, i = threadIdx.x >> 6;
    const int rest = blockIdx.x / (8 * FQ), wave = blockIdx.x / FQ % 8, j = blockIdx.x % FQ;
    int tp, tq;
    tile_at(job, job.whole + rest, tp, tq);
    const f32x4_t* from = reinterpret_cast<const f32x4_t*>(job.part) + ((long)blockIdx.x * 4 + i) * 64 + lane;
    const long stride = (long)R * 8 * 4 * FQ * 64;
    f32x4_t sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < job.split; s0 += 8) {
        f32x4_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = from[min(s0 + u, job.split - 1) * stride];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (s0 + u < job.split) {
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] = s0 + u == 0 ? v[u][e] : sum[e] + v[u][e];
            }
    }
    union { bf16_t h[4]; uint2 u; } o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o.h[e] = f32_to_bf16_bits(sum[e]);
    *reinterpret_cast<uint2*>(rows + (lane & 15) * TILE_PITCH + (i * 16 + (lane >> 4) * 4) * 2) = o.u;
    __syncthreads();
    if (threadIdx.x >= 128) return;
    const int row = threadIdx.x >> 3;
    const int m = tq * 32 * FQ + (wave >> 2) * (FQ * 16) + j * 16 + row, n = tp * TILE_N + (wave & 3) * 64 + (threadIdx.x & 7) * 8;
    if (m < job.M && n < job.N) store8<ACT>(job, m, n, *reinterpret_cast<const uint4*>(rows + row * TILE_PITCH + (threadIdx.x & 7) * 16));
}

template <int FQ, int ACT>
static int launch(const TileJob& job, hipStream_t s) {
    // (on every device: the attribute belongs to the device that is current)
    const hipError_t raised = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_tile_kernel<FQ, ACT>),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes(FQ));
    PTA_REQUIRE(raised == hipSuccess, "gemm_tile: %d bytes of LDS were refused", lds_bytes(FQ));
    const int R = job.tiles_p * job.tiles_q - job.whole;
    const int groups = (job.whole + 7) / 8 * 8 + (R * job.split + 7) / 8 * 8;
    hipLaunchKernelGGL((gemm_tile_kernel<FQ, ACT>), dim3(groups), dim3(512), lds_bytes(FQ), s, job);
    if (R > 0) hipLaunchKernelGGL((gemm_tile_reduce_kernel<FQ, ACT>), dim3(R * 8 * FQ), dim3(256), 0, s, job);
    return pta_check_launch("gemm_tile");
}

template <int ACT>
static int launch_fq(int fq, const TileJob& job, hipStream_t s) {
    switch (fq) {
        case 2: return launch<2, ACT>(job, s);
        case 3: return launch<3, ACT>(job, s);
        case 4: return launch<4, ACT>(job, s);
        case 5: return launch<5, ACT>(job, s);
        case 6: return launch<6, ACT>(job, s);
        case 7: return launch<7, ACT>(job, s);
        default: return launch<8, ACT>(job, s);
    }
}

static bool tile_sizes_ok(long M, long N, long K, long ldx) {
    return M > 0 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 && ldx % 8 == 0 && ldx >= K && (N + TILE_N) * K * 2 < TILE_PAST &&
           (M + 256) * ldx * 2 < TILE_PAST;
}

// How a product is shared out: 32 FQ rows of x a tile; the first `whole` tiles over all of K, the others in `split` ranges.
// What a choice takes, in microseconds, is put together from measurements (256 compute units):
//   a block of 64 elements of K, by FQ: `full` with every compute unit at work, `half` with at most half of them;
//   a tile's start and end: 2 + 0.55 FQ (first loads, results through LDS, the launch), from times at K = 1,024 to 8,192;
//   sums of cut tiles: 4.5 us for the second launch and 0.35 us a megabyte, written once and read once.
// The smallest sum wins.
struct TilePlan {
    int fq, whole, split;
    double us;
};

static TilePlan tile_plan(int M, int N, int K, int units) {
    static const double full[9] = {0, 0, 0.61, 0.69, 0.82, 0.95, 1.08, 1.25, 1.40};
    static const double half[9] = {0, 0, 0.67, 0.74, 0.78, 0.81, 0.90, 0.97, 1.07};
    const int blocks = (K + 63) / 64, tiles_p = (N + TILE_N - 1) / TILE_N;
    TilePlan best{0, 0, 1, 1e30};
    for (int fq = 2; fq <= 8; ++fq) {
        const long tiles = (long)tiles_p * ((M + 32 * fq - 1) / (32 * fq));
        auto block_us = [&](long groups) {
            const double busy = (double)groups / units;
            return busy >= 1.0 ? full[fq] : half[fq] + (full[fq] - half[fq]) * (busy > 0.5 ? 2.0 * busy - 1.0 : 0.0);
        };
        const double ends = 2.0 + 0.55 * fq;
        const long rounds = tiles / units, left = tiles % units;
        const double body = rounds * (blocks * full[fq] + ends);
        auto consider = [&](long whole, int split, double us) {
            if (us < best.us) best = TilePlan{fq, (int)whole, split, us};
        };
        consider(tiles, 1, body + (left ? blocks * block_us(left) + ends : 0.0));
        if (left == 0) continue;
        for (int split = 2; split <= 16 && split * 4 <= blocks; ++split) {
            const long groups = left * split;
            if (groups > 2L * units) break;
            const int each = (blocks + split - 1) / split;
            double us = body + 4.5 + 0.35 * groups * fq * 32768e-6;
            us += groups <= units ? each * block_us(groups) + ends : each * full[fq] + ends + each * block_us(groups - units) + ends;
            consider(rounds * units, split, us);
        }
    }
    return best;
}

extern "C" int pta_gemm_tile_plan(int M, int N, int K, int* fq, int* whole, int* split, long* part_values) {
    PTA_REQUIRE(tile_sizes_ok(M, N, K, K), "gemm_tile: M=%d N=%d K=%d: N and K must be multiples of 8, each matrix under 2 GiB", M, N, K);
    const TilePlan p = tile_plan(M, N, K, pta_compute_units());
    *fq = p.fq;
    *whole = p.whole;
    *split = p.split;
    const long tiles = (long)((N + TILE_N - 1) / TILE_N) * ((M + 32 * p.fq - 1) / (32 * p.fq));
    *part_values = (tiles - p.whole) * p.split * p.fq * 32 * TILE_N;
    return 0;
}

extern "C" int pta_gemm_tile_bf16(void* y, int ldy, const void* x, int ldx, const void* W, const float* bias, const void* add1,
                                  const void* add2, int M, int N, int K, int act, int fq, int whole, int split, float* part,
                                  long part_values, void* stream) {
    PTA_REQUIRE(y && x && W, "gemm_tile: null pointer");
    PTA_REQUIRE(tile_sizes_ok(M, N, K, ldx), "gemm_tile: M=%d N=%d K=%d ldx=%d: N, K and ldx must be multiples of 8, each matrix under 2 GiB", M, N, K, ldx);
    PTA_REQUIRE(ldy >= N && ldy % 8 == 0, "gemm_tile: rows of %d elements cannot lie %d apart (a multiple of 8)", N, ldy);
    for (const void* p : {(const void*)y, x, W, add1, add2, (const void*)part})
        PTA_REQUIRE(((uintptr_t)p % 16) == 0, "gemm_tile: pointers must be 16-byte aligned");
    PTA_REQUIRE(fq >= 2 && fq <= 8, "gemm_tile: a tile has 64 to 256 rows of x, got 32 x %d", fq);
    const long tiles_q = (M + 32L * fq - 1) / (32L * fq), tiles_p = (N + TILE_N - 1) / TILE_N, tiles = tiles_p * tiles_q;
    PTA_REQUIRE(whole >= 0 && whole <= tiles, "gemm_tile: %d of %ld tiles over all of K", whole, tiles);
    PTA_REQUIRE(split >= 1 && split <= (K + 63) / 64, "gemm_tile: %d ranges of %d blocks of K", split, (K + 63) / 64);
    const long rest = tiles - whole;
    PTA_REQUIRE(tiles * 8 * fq * split < (1L << 31), "gemm_tile: too many tiles (%ld) for one launch", tiles);
    PTA_REQUIRE(rest == 0 || (part && part_values >= rest * split * fq * 32 * TILE_N), "gemm_tile: room for %ld sums, %ld are needed",
                part_values, rest * split * fq * 32 * TILE_N);
    const TileJob job{(bf16_t*)y, part, (const bf16_t*)x, (const bf16_t*)W, bias, (const bf16_t*)add1, (const bf16_t*)add2,
                      M, N, K, ldx, ldy, (int)tiles_q, (int)tiles_p, whole, split};
    hipStream_t s = (hipStream_t)stream;
    switch (act) {
        case PTA_ACT_NONE: return launch_fq<PTA_ACT_NONE>(fq, job, s);
        case PTA_ACT_GELU: return launch_fq<PTA_ACT_GELU>(fq, job, s);
        case PTA_ACT_RELU2: return launch_fq<PTA_ACT_RELU2>(fq, job, s);
        default: return pta_fail("gemm_tile: activation %d is not applied here", act);
    }
}
