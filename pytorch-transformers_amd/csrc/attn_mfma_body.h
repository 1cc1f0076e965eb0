// What a workgroup of the attention kernel does (attn_mfma_impl.h), as text, because a launch of another kind carries it too
// (gemm_splitk_attn.hip) and the compiler did not survive it as a function at every head size.  Which workgroup it is stands in ATTN_X (of ATTN_NX),
// ATTN_Y and ATTN_Z; ATTN_INSIDE: it is part of a launch of another kind.
    constexpr int D = DT * 16;
    int window = 0, chunk = 0;  // chunk: blocks of positions that a token does not see out of (0: none)
    if constexpr (WIN) {
        ATTN_LATE(more);
        window = more.window_arg, chunk = more.chunk_arg;
    }
    // the lowest key that a token at position t sees: never decreasing in t
    auto lowest_key = [&](int t) {
        int lo = window > 0 ? max(0, t - window + 1) : 0;
        if (chunk > 0) lo = max(lo, t / chunk * chunk);
        return lo;
    };
    auto token_of = [&](int col) { return KS > 1 || ATTN_INSIDE ? 0 : col / g; };  // (launches for one token a sequence)
    constexpr int DS = (DT + 1) / 2;   // 32-wide steps over the head dimension
    constexpr int CHUNKS = D / 8;      // 16-byte chunks in a row of d elements
    static_assert(KS == 1 || W == 1, "waves either share key blocks or divide them");
    const int lane = threadIdx.x & 63, c = lane & 15, gq = lane >> 4;
    const int wave = KS > 1 || ATTN_INSIDE ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // which columns of the workgroup
    const int kw = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;     // which blocks of the keys
    // Ranges of keys are handed out range-major: the first ranges of every sequence, which all of them have whole,
    // start first, and the last ones, which are short or empty for most sequences, fill the launch's end.  (Sequence-
    // major, 32 sequences of 16,405 keys in ranges of 1,024 left two whole ranges to start when the first ones ended:
    // 45.8 us against 30.3 us at 16,384 keys.)
    int seq = ATTN_Z, split = 0, range0 = 0, range1 = 0;
    if (many_ranges) {
        ATTN_LATE(more);
        seq = ATTN_Z % more.n_seqs, split = ATTN_Z / more.n_seqs, range0 = split * more.split_size, range1 = range0 + more.split_size;
    }
    const int kvh = ATTN_Y;
    // The pages of a lone wave's first two blocks are looked up beside the sequence's length, not behind it: one round trip less in
    // a decode step's chain of them (an entry past the sequence's pages is read but not used).
    const int* bt = block_table + (long)seq * bt_stride;
    const int first_key = range0 + 32 * kw;
    int first_page = 0, next_page = 0;
    if constexpr (W == 1 && !WIN) {
        first_page = bt[min(first_key >> 6, bt_stride - 1)];
        next_page = bt[min((first_key + 32 * KS) >> 6, bt_stride - 1)];
    }
    int t0 = cu_tokens[seq], t1 = cu_tokens[seq + 1], start = seq_start[seq];
    if constexpr (W == 1 && !WIN) {
        // (behind another part of a launch, which writes memory, the entries come by vector loads)
        if constexpr (ATTN_INSIDE) first_page = __builtin_amdgcn_readfirstlane(first_page), next_page = __builtin_amdgcn_readfirstlane(next_page);
        else asm volatile("" : "+s"(first_page), "+s"(next_page), "+s"(t0), "+s"(t1), "+s"(start));
    }
    const int n_new = t1 - t0;
    const int ncols = n_new * g, n_groups = (ncols + 16 * CT * W - 1) / (16 * CT * W);
    // Column groups are handed out last first: late tokens see the most keys, and the longest work should
    // start first so that the launch ends evenly.  A paired launch has half the workgroups, and each takes a
    // late group and then the early group that mirrors it: under the causal mask the two together see as
    // many keys as any other pair, so a launch whose workgroups are all resident at once ends evenly too.
    for (int pass = 0; pass <= paired; ++pass) {
    int group = (W > 1 ? (int)ATTN_NX : n_groups) - 1 - (int)ATTN_X;  // (a sequence with fewer groups than the launch has room for: none below 0)
    if (paired) {
        const int late = n_groups - 1 - (int)ATTN_X, early = (int)ATTN_X;
        if (late < early || (pass == 1 && late == early)) return;
        group = pass == 0 ? late : early;
    }
    const int wg_col0 = group * (16 * CT * W);
    if (wg_col0 >= ncols || wg_col0 < 0) return;
    const int col0 = wg_col0 + wave * (16 * CT);
    const bool active = col0 < ncols;  // W > 1: a wave past the last column still loads and waits with the others
    const int last_col = min(ncols, col0 + 16 * CT) - 1;
    const int max_qpos = start + token_of(last_col);
    const int kv_len = start + n_new;
    // with a window a column at position t sees keys t - window + 1 .. t; this wave starts at the block of
    // the first key its first column sees (earlier pages may be gone), and at its range's start if split
    const int lo_first = WIN ? lowest_key(start + token_of(col0)) : 0;   // lowest key any column sees
    const int lo_last = WIN ? lowest_key(max_qpos) : 0;            // lowest key the last column sees
    const int k_begin = WIN ? max(range0, lo_first & ~31) : range0;
    const int k_end = !active ? 0 : many_ranges ? min(max_qpos + 1, range1) : max_qpos + 1;
    // below this key index no column of this wave masks anything (columns are ordered by token)
    const int min_lim = min(start + token_of(col0) + 1, k_end);
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
    // in the last 32-wide step of an odd number of 16-wide tiles, the upper half of the lanes has no data
    const uint32_t tail_keep = (DT % 2 == 1 && (DS - 1) * 4 + gq >= CHUNKS) ? 0u : 0xffffffffu;

    int qpos[CT], tok[CT], head[CT];
    float slope[CT];
    AFrag qf[CT][DS];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int col = col0 + ct * 16 + c;
        const int colc = min(col, ncols - 1);
        const int t = token_of(colc);
        tok[ct] = t0 + t;
        head[ct] = kvh * g + colc - t * g;
        qpos[ct] = col < ncols ? start + t : -1;  // -1: every key is masked for a column that does not exist
        const bf16_t* qp = q + ((long)tok[ct] * nh + head[ct]) * D;
#pragma unroll
        for (int ds = 0; ds < DS; ++ds) {
            const int chunk = ds * 4 + gq;
            qf[ct][ds].u = *reinterpret_cast<const uint4*>(qp + min(chunk, CHUNKS - 1) * 8);
            if (W > 1 && chunk >= CHUNKS) qf[ct][ds].u = zero4;
        }
    }

    // The sum of a column's weights is one more product: a tile of ones in the place of the values adds the
    // block's (rounded) weights of every column into lacc, whose sixteen rows all hold the same sums.  The
    // vector units, which bound this kernel, are spared eight additions a tile; the matrix cores take a ninth
    // instruction beside eight.
    f32x4_t oacc[DT][CT], lacc[CT];
    float m_run[CT], m_raise[CT];  // m_raise: the raw score above which the running maximum is brought up
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        m_run[ct] = -INFINITY;
        m_raise[ct] = -INFINITY;
        lacc[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) oacc[dt][ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    AFrag ones;
    ones.u = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);

    // AL says at compile time whether there is ALiBi (0: none, 1: there is; 2: whatever the launch brings), so
    // that the kernels for prompts, which are bound by their instruction stream, branch on nothing in it.
    // Scores are kept in units of log 2 (the scale carries log2 e), so that the exponential is the hardware's
    // exp2.  Without ALiBi the products are left unscaled, and the scale rides in the one multiply-add in front
    // of the exponential: s_mul is what a settled score is still to be multiplied by (positive).
    // What none of a lone wave's first loads of keys hangs on is read behind them.
    const float *slopes = nullptr, *sink = nullptr;
    float scale = 0.f, alibi_mul = 0.f, s_mul = 1.f;
    int bias_mode = 0, ranges = 1;
    bool has_alibi = AL == 1;
    bf16_t* out = nullptr;
    float *po = nullptr, *pm = nullptr, *pl = nullptr;
    PtaHeadRows rows;
    auto read_more = [&]() {
        ATTN_LATE(more);
        slopes = more.slopes, sink = more.sink, scale = more.scale, alibi_mul = more.alibi_mul, bias_mode = more.bias_mode, ranges = more.ranges;
        out = more.out, po = more.po, pm = more.pm, pl = more.pl;
        rows.ld = more.rows.ld, rows.head = more.rows.head, rows.keep = more.rows.keep, rows.mult = more.rows.mult;
        if (AL == 2) has_alibi = slopes != nullptr;
        s_mul = has_alibi ? 1.0f : scale;
        const float* of = slopes ? slopes : reinterpret_cast<const float*>(q);  // (a launch without slopes reads something and leaves it)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) slope[ct] = of[head[ct]];
    };
    constexpr bool FIRST = W > 1 || WIN || CT > 2;  // (of several tiles the registers run short, and these words would be kept in them all the while)
    if constexpr (FIRST) read_more();

    // The work on a block of 32 keys, in the four pieces that the loops below put together:
    // the products S^T = K . Q^T of the block, raw
    auto scores = [&](const AFrag (&k)[2][DS], f32x4_t (&sacc)[2][CT]) {
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
            AFrag k_last = k[tt][DS - 1];
            if (DT % 2 == 1) {
                k_last.u.x &= tail_keep; k_last.u.y &= tail_keep; k_last.u.z &= tail_keep; k_last.u.w &= tail_keep;
            }
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
                AFrag q_last = qf[ct][DS - 1];
                if (W == 1 && DT % 2 == 1) {  // (where q is loaded, a lone wave would wait for it before it asks for the first keys)
                    q_last.u.x &= tail_keep; q_last.u.y &= tail_keep; q_last.u.z &= tail_keep; q_last.u.w &= tail_keep;
                }
#pragma unroll
                for (int ds = 0; ds < DS; ++ds)
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ds == DS - 1 ? k_last.v : k[tt][ds].v, ds == DS - 1 ? q_last.v : qf[ct][ds].v, acc, 0, 0, 0);
                sacc[tt][ct] = acc;
            }
        }
    };
    // what the products become before the exponentials: with ALiBi, scaled and biased; keys that a column does
    // not see set to -inf; and the column's running maximum looked after.  MASKED = false is for a block that
    // every column of the wave sees whole: no key of it is past the sequence's end, past a column's own position
    // or before its window, and the code that would look is not there.
    auto settle = [&](auto masked_tag, f32x4_t (&sacc)[2][CT], int kb, float (&mx)[CT]) {
        constexpr bool MASKED = decltype(masked_tag)::value;
        const bool interior = !MASKED || (kb + 32 <= min_lim && kb >= lo_last);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            if (has_alibi) {  // one branch for the tile, not one per score
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int key = kb + 8 * gq + j;  // j = 4*tt + e
                    // the slope times the key's position, rounded as the reference rounds it (0) or exact (1), or
                    // times the key's distance from the query (2)
                    const float bias = bias_mode == 0 ? round_to_bf16(slope[ct] * round_to_bf16((float)key))
                                                      : slope[ct] * (float)(bias_mode == 2 ? key - qpos[ct] : key);
                    sacc[j >> 2][ct][j & 3] = sacc[j >> 2][ct][j & 3] * scale + bias * alibi_mul;
                }
            }
            if (MASKED && !interior) {
                const int lim = min(qpos[ct] + 1, k_end);  // keys below this, and from `lo` on, count for the column
                const int lo = WIN ? lowest_key(max(qpos[ct], 0)) : 0;
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (kb + 8 * gq + j >= lim || kb + 8 * gq + j < lo) sacc[j >> 2][ct][j & 3] = -INFINITY;
            }
            const f32x4_t s0 = sacc[0][ct], s1 = sacc[1][ct];
            constexpr bool PLAIN = W == 1 && CT == 4 && DT == 8;
            const float mx3 = max3<PLAIN>(s1[2], s1[3], max3<PLAIN>(s0[0], s0[1], s0[2]));
            mx[ct] = max3<PLAIN>(s0[3], s1[0], s1[1]);
            mx[ct] = max3<PLAIN>(mx[ct], mx3, mx3);
        }
    };
    // The running maximum is only a reference point for the exponentials, shared by the four lanes of a column;
    // it is brought up to the true maximum (an exchange between those lanes, and a rescale of what was summed)
    // only when some score of the block lies more than 2^8 above it, which after the first blocks of a row is
    // rare.  Weights stay below 2^8 and their rounding to bfloat16 is relative, so nothing is lost by a
    // reference that lags.  mx: the largest settled score of each tile's block, per lane.
    auto raise = [&](const float (&mx)[CT]) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            if (!__any(mx[ct] > m_raise[ct])) continue;
            float m = mx[ct] * s_mul;
            m = column_max(m);
            const float m_new = fmaxf(m_run[ct], m);
            const float corr = __builtin_amdgcn_exp2f(m_run[ct] - (m_new == -INFINITY ? 0.f : m_new));
            lacc[ct][0] *= corr;  // the one row of the sums that is read at the end
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                oacc[dt][ct][0] *= corr; oacc[dt][ct][1] *= corr; oacc[dt][ct][2] *= corr; oacc[dt][ct][3] *= corr;
            }
            m_run[ct] = m_new;
            m_raise[ct] = (m_new + 8.0f) / s_mul;
        }
    };
    // the weights 2^(score - reference) of the block, rounded, as the second product's operand
    auto weights = [&](const f32x4_t (&sacc)[2][CT], AFrag (&pf)[CT]) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const float m_use = m_run[ct] == -INFINITY ? 0.f : m_run[ct];
            float p[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[j >> 2][ct][j & 3], s_mul, -m_use));
            pf[ct].u = make_uint4(pack_bf16(p[0], p[1]), pack_bf16(p[2], p[3]), pack_bf16(p[4], p[5]), pack_bf16(p[6], p[7]));
        }
    };
    // sums of weights and O^T += V^T . P^T
    auto values = [&](const AFrag (&v)[DT], const AFrag (&pf)[CT]) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
            lacc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones.v, pf[ct].v, lacc[ct], 0, 0, 0);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
                oacc[dt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[dt].v, pf[ct].v, oacc[dt][ct], 0, 0, 0);
    };
    // four neighbours of a result (inside a launch of another kind other dies read them in the same launch: through to the memory they share)
    auto store4 = [&](bf16_t* to, uint2 v) {
        if constexpr (ATTN_INSIDE)
            __hip_atomic_store(reinterpret_cast<unsigned long long*>(to), (unsigned long long)v.y << 32 | v.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *reinterpret_cast<uint2*>(to) = v;
    };
    const std::true_type masked_block;
    const std::false_type whole_block;
    // a key whose index is not below lim is taken out of eight values of consecutive keys from kbase on
    auto keep_below = [&](uint4& v, int kbase, int lim) {
        uint32_t mk[4];
#pragma unroll
        for (int w = 0; w < 4; ++w)
            mk[w] = (kbase + 2 * w < lim ? 0x0000ffffu : 0u) | (kbase + 2 * w + 1 < lim ? 0xffff0000u : 0u);
        v.x &= mk[0]; v.y &= mk[1]; v.z &= mk[2]; v.w &= mk[3];
    };

    if constexpr (W == 1) {
        // all of a block at once
        auto use_block = [&](KvBlock<DT>& b, int kb) {
            if (kb + 32 > kv_len) {
                // positions past the sequence's end were never written; whatever lies there must not reach the
                // sum, not even with weight zero
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) keep_below(b.v[dt].u, kb + gq * 8, kv_len);
            }
            f32x4_t sacc[2][CT];
            AFrag pf[CT];
            float mx[CT];
            scores(b.k, sacc);
            settle(masked_block, sacc, kb, mx);
            raise(mx);
            weights(sacc, pf);
            values(b.v, pf);
        };
        // Two register buffers: while one block is used, the loads of the next are in flight (a wave alone has nothing else to hide
        // the memory's latency behind), and what is not used is not asked for: a block loaded past the wave's last costs as
        // much as one that counts (launches over cold caches, us, the next block always loaded -> only where there is one: 13 heads on
        // 13 of 80, 5 sequences of 40 / 210 / 320 keys 6.2 -> 5.5, 8.1 -> 6.9, 9.4 -> 8.3; 71 on 1 of 64, 8 of 100 6.0 -> 5.1; 32 on 8 of 128, 32 of
        // 100 / 270 10.3 -> 7.8, 13.2 -> 12.2).  The loads stand in straight lines of code, not behind
        // conditions: where ways with and without a load meet, the compiler waits for all of them.
        constexpr int STEP = 32 * KS;  // from one block of this wave to its next
        KvBlock<DT> b0, b1;
        const int k_first = k_begin + 32 * kw;
        const int n_mine = k_first < k_end ? (k_end - k_first + STEP - 1) / STEP : 0;  // blocks of this wave
        auto blk = [&](int j) { return k_first + STEP * j; };
        auto page_of = [&](int kb) {
            if constexpr (!WIN) {
                if (kb >> 6 == first_key >> 6) return (long)first_page;
                if (kb >> 6 == (first_key + STEP) >> 6) return (long)next_page;
            }
            return (long)bt[kb >> 6];
        };
        auto load = [&](KvBlock<DT>& to, int j) {
            load_block<DT>(to, blk(j), page_of(blk(j)), k_pool, v_pool, nkv, kvh, c, gq);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto use = [&](KvBlock<DT>& from, int j) {
            use_block(from, blk(j));
            __builtin_amdgcn_sched_barrier(0);
        };
        if (n_mine > 0) {
            load(b0, 0);
            if constexpr (!FIRST) read_more();
            int j = 0;
            for (; j + 2 < n_mine; j += 2) {
                load(b1, j + 1);
                use(b0, j);
                load(b0, j + 2);
                use(b1, j + 1);
            }
            if (j + 1 < n_mine) {
                load(b1, j + 1);
                use(b0, j);
                b0 = b1;
                ++j;
            }
            use(b0, j);
        } else if constexpr (!FIRST) read_more();
    } else {
        // The workgroup's waves walk the keys of its last column together, a stage of SK keys (one or two
        // blocks) between barriers.  A stage goes global memory -> registers (one stage ahead) -> one of two
        // LDS buffers -> each wave's operand registers.  Key rows are stored in the order the score tiles want
        // them (within a block: tile tt, lane column c <-> key 8*(c/4) + 4*tt + c%4), so that sixteen lanes
        // read sixteen consecutive LDS rows; the row strides (D*2 + 16 and SK*2 + 16 bytes) put those on
        // distinct banks.  Small heads take a whole page per stage: half the barriers.
        constexpr int SK = D <= 64 ? 64 : 32, NBK = SK / 32;
        constexpr int KROW = D + 8, VROW = SK + 8;                // elements
        constexpr int KPIECES = SK / 8 * D, THREADS = 64 * W;     // 16-byte pieces of a stage's keys (and values)
        constexpr int PER = (KPIECES + THREADS - 1) / THREADS;
        constexpr int VCH = SK / 8;                               // pieces in a stage's row of values
        __shared__ __attribute__((aligned(16))) bf16_t kbuf[2][SK * KROW];
        __shared__ __attribute__((aligned(16))) bf16_t vbuf[2][D * VROW];
        const int tid = threadIdx.x;
        const int wg_last_col = min(ncols, wg_col0 + 16 * CT * W) - 1;
        // (a launch that cuts the keys into ranges walks its own range only)
        const int k_end_wg = many_ranges ? min(start + wg_last_col / g + 1, range1)
                                          : start + wg_last_col / g + 1;
        const int k_begin_wg = max(WIN ? lowest_key(start + wg_col0 / g) & ~(SK - 1) : 0,
                                   range0);
        const int ks_last = (kv_len - 1) & ~(SK - 1);  // the last stage that has a page
        static_assert(PER <= 2, "a thread moves at most two pieces of keys and two of values per stage");
        static_assert(PTA_PAGE % SK == 0, "a stage lies in one page");
        // the pieces in flight are plain variables, not an array: an array that lambdas index stays in
        // scratch memory at the larger head sizes, and every stage then waits for its loads at once
        uint4 gk0, gk1, gv0, gv1;
        const int p0 = min(tid, KPIECES - 1), p1 = min(tid + THREADS, KPIECES - 1);
        auto gload = [&](int ks) {  // keys and values of the stage at ks (clamped to the last one there is)
            ks = min(ks, ks_last);
            const long page = ((long)bt[ks >> 6] * nkv + kvh) * (long)(PTA_PAGE * D);
            const bf16_t* kpage = k_pool + page + (long)(ks & 63) * D;
            const bf16_t* vpage = v_pool + page + (ks & 63);
            gk0 = *reinterpret_cast<const uint4*>(kpage + (long)(p0 / CHUNKS) * D + (p0 % CHUNKS) * 8);
            gv0 = *reinterpret_cast<const uint4*>(vpage + (long)(p0 / VCH) * PTA_PAGE + (p0 % VCH) * 8);
            if constexpr (PER > 1) {
                gk1 = *reinterpret_cast<const uint4*>(kpage + (long)(p1 / CHUNKS) * D + (p1 % CHUNKS) * 8);
                gv1 = *reinterpret_cast<const uint4*>(vpage + (long)(p1 / VCH) * PTA_PAGE + (p1 % VCH) * 8);
            }
        };
        // Positions past the sequence's end were never written; whatever lies there must not reach the sums, not
        // even with weight zero: such values are cleared on their way into LDS.
        auto put = [&](int buf, int p, const uint4& k, uint4 v, int ks) {
            if (p < KPIECES) {
                const int kk = p / CHUNKS;  // key of the stage -> its row in operand order
                const int row = (kk & ~31) + ((kk & 7) >> 2) * 16 + 4 * ((kk & 31) >> 3) + (kk & 3);
                *reinterpret_cast<uint4*>(&kbuf[buf][row * KROW + (p % CHUNKS) * 8]) = k;
                if (ks + SK > kv_len) keep_below(v, ks + (p % VCH) * 8, kv_len);
                *reinterpret_cast<uint4*>(&vbuf[buf][(p / VCH) * VROW + (p % VCH) * 8]) = v;
            }
        };
        auto sstore = [&](int ks) {  // into the buffer of the stage's number, whatever was loaded for it
            const int buf = (ks / SK) & 1;
            put(buf, tid, gk0, gv0, min(ks, ks_last));
            if constexpr (PER > 1) put(buf, tid + THREADS, gk1, gv1, min(ks, ks_last));
        };
        auto lfetch_k = [&](AFrag (&k)[2][DS], int kb) {  // the keys of the block at kb, from its stage's buffer
            const bf16_t* kb_lds = &kbuf[(kb / SK) & 1][((kb & (SK - 1)) + c) * KROW];
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int ds = 0; ds < DS; ++ds)
                    k[tt][ds].u = *reinterpret_cast<const uint4*>(kb_lds + tt * 16 * KROW + min(ds * 4 + gq, CHUNKS - 1) * 8);
        };
        auto lfetch_v = [&](AFrag (&v)[DT], int kb) {
            const bf16_t* vb_lds = &vbuf[(kb / SK) & 1][c * VROW + (kb & (SK - 1)) + gq * 8];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) v[dt].u = *reinterpret_cast<const uint4*>(vb_lds + dt * 16 * VROW);
        };
        gload(k_begin_wg);
        sstore(k_begin_wg);
        __syncthreads();
        for (int ks = k_begin_wg; ks < k_end_wg; ks += SK) {
            gload(ks + SK);
            __builtin_amdgcn_sched_barrier(0);
            // the blocks of the stage that are this wave's: a plain loop with one way through it, in which the
            // compiler leaves the sums in their registers (two copies of the block's second half, one for the
            // rare block that raises a maximum, made it move all of them in every block)
            const int b_hi = min(ks + SK, k_end);
            for (int kb = max(ks, k_begin); kb < b_hi; kb += 32) {
                f32x4_t sacc[2][CT];
                AFrag pf[CT], kf[2][DS], vf[DT];
                float mx[CT];
                lfetch_k(kf, kb);
                scores(kf, sacc);
                if (kb + 32 <= min_lim && kb >= lo_last) settle(whole_block, sacc, kb, mx);
                else settle(masked_block, sacc, kb, mx);
                raise(mx);
                weights(sacc, pf);
                lfetch_v(vf, kb);
                values(vf, pf);
            }
            __builtin_amdgcn_sched_barrier(0);
            sstore(ks + SK);
            __syncthreads();
        }
    }

    if constexpr (KS > 1) {
        // every wave's sums, running maxima and unnormalised results go to LDS; then the (column tile, feature
        // tile) pairs are dealt out to the waves, and each merges its pairs over the waves in their order
        extern __shared__ __attribute__((aligned(16))) float ks_mem[];
        float4* so = reinterpret_cast<float4*>(ks_mem);
        float* sm = ks_mem + KS * CT * DT * 256;
        float* sl = sm + KS * CT * 16;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const float l = lacc[ct][0];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                so[((kw * CT + ct) * DT + dt) * 64 + lane] =
                    make_float4(oacc[dt][ct][0], oacc[dt][ct][1], oacc[dt][ct][2], oacc[dt][ct][3]);
            if (gq == 0) {
                sm[(kw * CT + ct) * 16 + c] = m_run[ct];
                sl[(kw * CT + ct) * 16 + c] = l;
            }
        }
        __syncthreads();
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            float mx = -INFINITY, l = 0.f, wgt[KS];
#pragma unroll
            for (int w = 0; w < KS; ++w) wgt[w] = sm[(w * CT + ct) * 16 + c];
#pragma unroll
            for (int w = 0; w < KS; ++w) mx = fmaxf(mx, wgt[w]);
#pragma unroll
            for (int w = 0; w < KS; ++w) {
                wgt[w] = wgt[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(wgt[w] - mx);
                l += wgt[w] * sl[(w * CT + ct) * 16 + c];
            }
            if (sink && !many_ranges) l += __builtin_amdgcn_exp2f(sink[head[ct]] * PTA_LOG2E - mx);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                if ((ct * DT + dt) % KS != kw || qpos[ct] < 0) continue;
                float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int w = 0; w < KS; ++w) {
                    const float4 o = so[((w * CT + ct) * DT + dt) * 64 + lane];
                    acc.x += wgt[w] * o.x; acc.y += wgt[w] * o.y; acc.z += wgt[w] * o.z; acc.w += wgt[w] * o.w;
                }
                const long row = (long)tok[ct] * nh + head[ct];
                if (!many_ranges) {
                    const float inv = rows.mult / l;
                    uint2 w2;
                    w2.x = pack_bf16(acc.x * inv, acc.y * inv);
                    w2.y = pack_bf16(acc.z * inv, acc.w * inv);
                    if (dt * 16 + gq * 4 < rows.keep)
                        store4(out + (long)tok[ct] * rows.ld + (long)head[ct] * rows.head + dt * 16 + gq * 4, w2);
                } else {
                    *reinterpret_cast<float4*>(po + (row * ranges + split) * D + dt * 16 + gq * 4) = acc;
                    if (dt == 0 && gq == 0) {
                        pm[row * ranges + split] = mx;
                        pl[row * ranges + split] = l;
                    }
                }
            }
        }
    } else {
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        float l = lacc[ct][0];
        if (qpos[ct] < 0) continue;
        const long row = (long)tok[ct] * nh + head[ct];
        if (!many_ranges) {
            if (sink) l += __builtin_amdgcn_exp2f(sink[head[ct]] * PTA_LOG2E - m_run[ct]);
            const float inv = rows.mult / l;
            bf16_t* o = out + (long)tok[ct] * rows.ld + (long)head[ct] * rows.head;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                uint2 w;
                w.x = pack_bf16(oacc[dt][ct][0] * inv, oacc[dt][ct][1] * inv);
                w.y = pack_bf16(oacc[dt][ct][2] * inv, oacc[dt][ct][3] * inv);
                if (dt * 16 + gq * 4 < rows.keep) store4(o + dt * 16 + gq * 4, w);
            }
        } else {
            // a range past the column's keys has nothing to add: only its marker is written, and the combine
            // does not read past the last range that has one.  A range before a window is followed by ranges
            // that count, so it is read with weight zero and must hold numbers: the (zero) sums are written.
            if (k_begin < k_end || WIN) {
                float* o = po + (row * ranges + split) * D;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
                    *reinterpret_cast<float4*>(o + dt * 16 + gq * 4) =
                        make_float4(oacc[dt][ct][0], oacc[dt][ct][1], oacc[dt][ct][2], oacc[dt][ct][3]);
            }
            if (gq == 0) {
                pm[row * ranges + split] = m_run[ct];
                pl[row * ranges + split] = l;
            }
        }
    }
    }
    }  // pass
