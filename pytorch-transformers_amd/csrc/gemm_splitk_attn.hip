// A decode step's attention and both products that end a block, the feed-forward's (a) and the attention's output product (b), in one
// launch: partial sums of x1 . W1^T and x2 . W2^T as pta_gemm_splitk_pair_bf16 leaves them, with x2 = attention.
//
// Attention of a short context is a chain of a few loads on a few workgroups, some 5 us in which next to nothing comes from memory, and the
// larger product, of 165 MB at 7B sizes, has no need of it.  So the launch begins with the attention's workgroups, goes on with those of a,
// which start at once, and ends with those of b, which ask for their first rows of W and then wait until all of attention is done, as
// it then long is.
//
// Attention, the pair and the norm behind it, us, launches apart -> this: 4,544 x 18,176 with 71 heads on one KV head, 1 / 8 / 16 / 32 sequences of 150 keys
// 48.6 -> 45.5, 49.6 -> 47.5, 50.9 -> 49.2, 54.1 -> 52.4 (a wave on a piece's keys), 1 and 8 of 1,900 51.7 -> 46.1, 55.3 -> 50.3 (four waves, and
// no merge of ranges); the attention alone takes 4.7 to 8 us there, the merge 4.4.  What is lost of it are the places that attention's workgroups have on
// the compute units, each for a chain of loads that wait behind the stream: many pieces ride no longer, nor any where both
// products keep a unit about as long, which then ends with the attention instead of beside it (tuning.py has both lines).
//
// The wait ends whatever order workgroups start in: one that has looked for a while does what of attention it does not find done itself, which
// writes the values that stand there or will.
//
// Results change hands in the memory that all dies share: attention's are stored through to it, a workgroup marks its worth of attention as
// done once its stores have arrived, and x2 is asked for once all marks have been seen.  No cache holds older values of x2: nothing of it is read earlier in
// the launch, and caches are empty of other launches' data when one starts.
#include "gemm_splitk_attn.h"

#define PATIENCE 4096  // looks at the marks, a microsecond or two each, before a workgroup does pieces itself

__device__ __forceinline__ bool is_done(const int* mark) { return __hip_atomic_load(mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0; }

struct RideGate {
    static constexpr bool closed = true;
    const AttnRide& ride;
    int* seen;
    __device__ __forceinline__ bool wait(bool second) const {
        if (!second) return true;
        if (threadIdx.x < 64) {
            bool all = false;
            for (int n = 0; n < PATIENCE && !all; ++n) {
                bool mine = true;
                for (int t = threadIdx.x; t < ride.tasks; t += 64) mine &= is_done(ride.sync + t);
                all = __all(mine);
            }
            if (threadIdx.x == 0) *seen = all;
        }
        __syncthreads();
        const bool open = __builtin_amdgcn_readfirstlane(*seen) != 0;
        if (!open) wait_loads<0>();  // attention is to have the LDS that the first stages of W go to
        __syncthreads();
        return open;
    }
};

// sixteen heads of a KV head of a sequence
template <int DT, int CT, int W, bool WIN, int KS, int AL>
__device__ __forceinline__ void attend_to(const AttnArgs& a, int place_x, int place_y, int place_z, int groups) {
    const bf16_t *const q = a.q, *const k_pool = a.k_pool, *const v_pool = a.v_pool;
    const int *const block_table = a.block_table, *const cu_tokens = a.cu_tokens, *const seq_start = a.seq_start;
    const int bt_stride = a.bt_stride, nh = a.nh, nkv = a.nkv, g = nh / nkv;
    constexpr int paired = 0;
    constexpr bool many_ranges = false;
#define ATTN_X place_x
#define ATTN_Y place_y
#define ATTN_Z place_z
#define ATTN_NX groups
#define ATTN_INSIDE 1
#define ATTN_LATE(more) const AttnMore& more = a.more
#include "attn_mfma_body.h"
#undef ATTN_X
#undef ATTN_Y
#undef ATTN_Z
#undef ATTN_NX
#undef ATTN_INSIDE
#undef ATTN_LATE
}

// workgroup t's worth of pieces; KS: waves that share a piece's keys
template <int KS>
__device__ __forceinline__ void attend(const AttnRide& ride, int t) {
    const int piece = KS > 1 ? t : t * RIDE_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), rest = piece / ride.groups;
    if (rest < ride.attn.nkv * ride.n_seqs)
        attend_to<RIDE_HEAD, 1, 1, false, KS, 2>(ride.attn, piece % ride.groups, rest % ride.attn.nkv, rest / ride.attn.nkv, ride.groups);
    wait_loads<0>();  // stores, too, are counted: this wave's have arrived
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(ride.sync + t, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int MT, int RT, bool ROT, int KS>
__global__ __launch_bounds__(SK_WAVES * 64, RT == 2 ? 1 : MT > 2 ? 2 : 3) void gemm_splitk_attn_kernel(SplitkProblem pa, SplitkProblem pb, int M,
                                                                                                   int rot_stride, AttnRide ride) {
    __shared__ int seen;
    if ((int)blockIdx.x < ride.owners) return attend<KS>(ride, blockIdx.x);
    const int block = (int)blockIdx.x - ride.owners, blocks = pa.tiles * pa.parts + pb.tiles * pb.parts;
    if (splitk_body<MT, RT, 4, ROT, SK_WAVES>(pa, pb, M, 1, M, rot_stride, block, blocks, RideGate{ride, &seen})) return;
    for (int t = 0; t < ride.tasks; ++t) {
        if (threadIdx.x == 0) seen = is_done(ride.sync + t);
        __syncthreads();
        const bool done = __builtin_amdgcn_readfirstlane(seen) != 0;
        __syncthreads();
        if (!done) attend<KS>(ride, t);
    }
    __syncthreads();
    splitk_body<MT, RT, 4, ROT, SK_WAVES>(pa, pb, M, 1, M, rot_stride, block, blocks, NoGate{});
}

template <int MT, int RT, int KS>
static int launch(const SplitkProblem& a, const SplitkProblem& b, int M, bool rotate, int rot_stride, const AttnRide& ride, hipStream_t s) {
    constexpr int stages = 4 * splitk_slot(MT, RT, SK_WAVES), keys = (int)key_split_lds(RIDE_HEAD, 1, KS), lds = stages > keys ? stages : keys;
    static_assert(lds <= 158 * 1024, "the stages must fit the LDS of a compute unit");
    auto kern = rotate ? gemm_splitk_attn_kernel<MT, RT, true, KS> : gemm_splitk_attn_kernel<MT, RT, false, KS>;
    if (lds > 60 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
        return pta_fail("gemm_splitk_pair_attn: cannot have %d bytes of LDS", lds);
    hipLaunchKernelGGL(kern, dim3(ride.owners + a.tiles * a.parts + b.tiles * b.parts), dim3(SK_WAVES * 64), lds, s, a, b, M, rot_stride, ride);
    return pta_check_launch("gemm_splitk_pair_attn");
}

template <int KS>
static int launch_rows(const SplitkProblem& a, const SplitkProblem& b, int M, int rows, bool rotate, int rot_stride, const AttnRide& ride, hipStream_t s) {
    switch ((M + 15) / 16) {
        case 1: return launch<1, 1, KS>(a, b, M, rotate, rot_stride, ride, s);
        case 2: return launch<2, 1, KS>(a, b, M, rotate, rot_stride, ride, s);
        case 3: return rows == 2 ? launch<3, 2, KS>(a, b, M, rotate, rot_stride, ride, s) : launch<3, 1, KS>(a, b, M, rotate, rot_stride, ride, s);
        default: return rows == 2 ? launch<4, 2, KS>(a, b, M, rotate, rot_stride, ride, s) : launch<4, 1, KS>(a, b, M, rotate, rot_stride, ride, s);
    }
}

int pta_splitk_attn_launch(const SplitkProblem& a, const SplitkProblem& b, int M, int rows, bool rotate, int rot_stride, bool share_keys,
                           const AttnRide& ride, hipStream_t s) {
    return share_keys ? launch_rows<RIDE_WAVES>(a, b, M, rows, rotate, rot_stride, ride, s) : launch_rows<1>(a, b, M, rows, rotate, rot_stride, ride, s);
}
