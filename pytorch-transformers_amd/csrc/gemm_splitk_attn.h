// The launch that carries a decode step's attention beside the two products of a block's end (gemm_splitk_attn.hip).
#pragma once

#include "attn_mfma_impl.h"
#include "gemm_splitk_impl.h"

#define RIDE_MOST_ROWS 64   // of x
#define RIDE_HEAD 4         // sixteens of a head
#define RIDE_WAVES 4        // of a workgroup

// attn_mfma_kernel's arguments for one token a sequence and whole contexts
struct AttnArgs {
    const bf16_t *q, *k_pool, *v_pool;
    const int *block_table, *cu_tokens, *seq_start;
    int bt_stride, nh, nkv;
    AttnMore more;
};

struct AttnRide {
    AttnArgs attn;
    int groups, n_seqs;  // pieces of attention: groups (sixteen heads of a KV head) x KV heads x sequences
    int tasks, owners;   // workgroups' worth of them, and how many of those the launch begins with
    int* sync;           // whether each is done; zeros when the launch starts
};

// a: a product of its own, b: that of what attention gives; `rows`: tiles of sixteen rows of W a wave (1 or 2);
// share_keys: a workgroup's four waves have a piece, and its keys block by block in turn, else four pieces, a wave each
int pta_splitk_attn_launch(const SplitkProblem& a, const SplitkProblem& b, int M, int rows, bool rotate, int rot_stride, bool share_keys,
                           const AttnRide& ride, hipStream_t s);
