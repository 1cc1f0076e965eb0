// Rows of a matrix straight to LDS, a wave by itself: what the kernels for few rows read their weights through.
//
// The matrix instruction wants a lane's operand to be sixteen bytes of row lane % 16.  Loaded that way, any sixteen neighbouring
// lanes touch sixteen rows, and the address path takes them one cache line a cycle: reading 207 MB so takes 48 us at best, where
// loads of whole 128-byte lines, eight lanes a line, take 38 to registers and 35 straight to LDS (5.9 TB/s; reading the array
// from end to end 33; rows of 16 KB: 680 MB in 149, 109 and 108 us).  So a wave's load brings eight rows by 128 bytes to LDS and the
// operands are read from there; each wave has a ring of its own and waits for its own loads, so there is no barrier.
//
// A row of a slot is 64 elements, 128 bytes without a gap: sixteen bytes c of row r lie at place c ^ (r / 2 % 8), so that any
// sixteen lanes that read together cover every bank once.  Each lane of a load asks for the sixteen bytes that its place is to hold.
#pragma once
#include "common.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

#define LDS_PAST 0x7ffffff0  // an offset past the end of every operand: such loads give zeros

// waits until at most N of the wave's loads are on their way
template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

__device__ __forceinline__ void wait_reads() { __builtin_amdgcn_s_waitcnt(0xc07f); }  // lgkmcnt(0)

// Sixteen bytes a lane from byte `at` of a buffer straight to LDS, one lane after the other from `to` on; zeros past the
// buffer's end.  Written out because the compiler would wait for every such load before any read of LDS; the waits are
// the kernels' own (wait_loads).  There is no register that the load writes.
__device__ __forceinline__ void fetch16(i32x4_t buffer, unsigned to, int at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(at), "s"(buffer) : "memory");
}

__device__ __forceinline__ i32x4_t buffer_of(const void* p, int bytes) {
    const uint64_t at = (uint64_t)(uintptr_t)p;
    return i32x4_t{__builtin_amdgcn_readfirstlane((int)(uint32_t)at), __builtin_amdgcn_readfirstlane((int)((uint32_t)(at >> 32) & 0xffffu)),
                   __builtin_amdgcn_readfirstlane(bytes), 0x00020000};
}

__device__ __forceinline__ unsigned lds_address(const char* p) { return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const char*)p; }

// which row of a tile of sixteen a lane asks for in the tile's load l (0, 1), and the first element of its sixteen bytes
__device__ __forceinline__ int stream_row(int lane, int l) { return l * 8 + (lane >> 3); }
__device__ __forceinline__ int stream_element(int lane, int l) { return ((lane & 7) ^ ((4 * l + (lane >> 4)) & 7)) * 8; }

// Elements of a row that this takes: the rows of a tile lie within 32-bit bytes of each other, those of a query_key_value
// projection's rotation pairs (up to 512 rows apart) too.
#define STREAM_MOST_K (1 << 20)

template <int LOADS>
struct RingTail {
    // the last steps, T + 1 of them if there are so many: each waits until only what is asked for behind it is on its way
    template <int T, typename Step>
    static __device__ __forceinline__ void last_steps(int n, Step step) {
        if (T < n) {
            wait_loads<T * LOADS>();
            step();
        }
        if constexpr (T > 0) last_steps<T - 1>(n, step);
    }
};

// RT tiles of sixteen rows of W and one of x, by steps of 64 elements of K: the wave takes the steps wave, wave + S, ..., D of
// them on their way at a time.  w: each tile's buffer; w_at, x_at: byte offsets of the lane's rows (stream_row) within their
// buffers, LDS_PAST for none.  The steps are walked from `rot` on, round.
template <int RT, int D>
struct RowStream {
    static constexpr int SLOT = (RT + 1) * 2048, RING = D * SLOT, LOADS = 2 * (RT + 1);
    i32x4_t w[RT], x;
    int w_at[2 * RT], x_at[2];

    // S: a power of two.  Loads are asked for as far as there are steps: the last D steps wait for fewer and fewer.
    __device__ __forceinline__ void run(f32x4_t (&acc)[RT], const char* ring, int lane, int any_wave, int S, int K, int nsteps, int rot) const {
        const unsigned to = __builtin_amdgcn_readfirstlane(lds_address(ring));
        const int wave = __builtin_amdgcn_readfirstlane(any_wave);
        const int c8[2] = {stream_element(lane, 0), stream_element(lane, 1)};
        auto issue = [&](int step, int slot) {
            int s = step + rot;
            s -= s >= nsteps ? nsteps : 0;
            const int k = s * 64;
#pragma unroll
            for (int l = 0; l < LOADS; ++l) {
                const int row_at = l < 2 * RT ? w_at[l] : x_at[l & 1];
                const int at = row_at != LDS_PAST && k + c8[l & 1] < K ? row_at + (k + c8[l & 1]) * 2 : LDS_PAST;
                fetch16(l < 2 * RT ? w[l >> 1] : x, to + slot + l * 1024, at);
            }
        };
        const int in_row = (lane & 15) * 128 + (((lane >> 4) ^ ((lane & 15) >> 1)) & 7) * 16;
        bf16x8_t a[2][RT + 1];
        auto read = [&](int slot) {
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int t = 0; t <= RT; ++t) a[hf][t] = *reinterpret_cast<const bf16x8_t*>(ring + ((in_row ^ (hf * 64)) + slot + t * 2048));
        };
        auto multiply = [&]() {
#pragma unroll
            for (int hf = 0; hf < 2; ++hf)
#pragma unroll
                for (int t = 0; t < RT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[hf][t], a[hf][RT], acc[t], 0, 0, 0);
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
    }
};
