"""The 32-bit kernels alone, against 64-bit references: every way a product runs (few rows, tiles, shared segments) and both
attention kernels, at the edges of their tiles, and the same bits for a row whichever of them it runs in."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from pytorch_transformers_amd import ops

    ops.load_library()
    return ops


def _rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).cuda()


@pytest.mark.parametrize("N,K", [(1, 1), (40, 15), (129, 16), (260, 100), (64, 1040), (4544, 576), (8200, 300), (96, 2050),
                                 (5376, 100), (5376, 48), (70, 1044)])
def test_products(N, K):
    """Rows 1 .. 700 (few rows with one, two and four tiles; 64 and, at 5376 columns, 128 tiles; shared segments), K with and without a last
    block and rows that are no multiple of sixteen bytes."""
    ops = _ops()
    M = 700
    a, w, bias, a1, a2 = _rand(M, K), _rand(N, K, seed=1), _rand(N, seed=2), _rand(M, N, seed=3), _rand(M, N, seed=4)
    prod = a.double() @ w.double().T
    # |error| <= K eps sum |a w| in the worst case; the sums are of random signs, so sqrt(K) eps times the root of the sum of squares
    scale = ((a.double() ** 2) @ (w.double() ** 2).T).sqrt().max().item()
    tol = 8 * 2.0 ** -24 * math.sqrt(K) * scale + 1e-30
    plain = ops.gemm_f32(a, w)
    assert (plain.double() - prod).abs().max().item() <= tol
    v = prod + bias.double()
    want = 0.5 * v * (1 + torch.erf(v / math.sqrt(2.0))) + a1.double() + a2.double()
    full = ops.gemm_f32(a, w, bias, "gelu", a1, a2)
    assert (full.double() - want).abs().max().item() <= 2 * tol + 2e-6 * want.abs().max().item()
    for m in (1, 2, 16, 17, 33, 64, 65, 128, 300):
        assert torch.equal(ops.gemm_f32(a[:m].contiguous(), w), plain[:m]), f"{m} rows alone and in a batch"
        assert torch.equal(ops.gemm_f32(a[:m].contiguous(), w, bias, "gelu", a1[:m].contiguous(), a2[:m].contiguous()), full[:m])


def _product_as(ops, a, w, fp, fq, whole, share):
    """The product by tiles of 64 ``fp`` rows of w by 32 ``fq`` rows of a (0: few rows), the first ``whole`` over all of K."""
    (M, K), N = a.shape, w.shape[0]
    out = torch.full((M, N), 7.0, device="cuda")
    scratch = torch.empty(16 << 20, dtype=torch.float32, device="cuda")
    ops._call("pta_gemm_f32_as", ops._ptr(out), ops._ptr(a), ops._ptr(w), ops._ptr(None), ops._ptr(None), ops._ptr(None), M, N, K, 0,
              fp, fq, whole, share, ops._ptr(scratch), ctypes.c_long(scratch.numel()), ops._stream())
    return out


def _split_tol(a, w):
    """What the sums in 32 bits may be off by: as test_products."""
    scale = ((a.double() ** 2) @ (w.double() ** 2).T.contiguous()).sqrt().max().item()
    return 8 * 2.0 ** -24 * math.sqrt(a.shape[1]) * scale + 1e-30


# K: no last block of 32; a last block; rows of sixteen bytes and not; fewer blocks than segments, as many, and more
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (33, 129, 32), (129, 257, 100), (64, 256, 256), (130, 70, 1044), (257, 300, 2050), (70, 520, 4544)])
@pytest.mark.parametrize("offset", [0, 1])
def test_products_by_every_way(M, N, K, offset):
    """Few rows, every size of tile, tiles over all of K, cut ones and both: the same bits, also off sixteen-byte addresses."""
    ops = _ops()
    a, w = (_rand(n * K + 1, seed=i)[offset:offset + n * K].view(n, K) for i, n in enumerate((M, N)))
    want = _product_as(ops, a, w, 0, 0, 0, 1)
    assert (want.double() - a.double() @ w.double().T).abs().max().item() <= _split_tol(a, w)
    blocks = -(-K // 32)
    segments = -(-blocks // -(-blocks // 8))
    for fp in (2, 4):
        for fq in (1, 2, 3, 4):
            tiles = -(-N // (64 * fp)) * -(-M // (32 * fq))
            for whole, share in {(tiles, 1), (0, 1), (0, segments), (tiles // 2, segments), (0, (segments + 1) // 2)}:
                assert torch.equal(_product_as(ops, a, w, fp, fq, whole, share), want), (fp, fq, whole, share)


def test_product_of_rows_that_tiles_cannot_address():
    """Rows too long for 32-bit offsets within a tile go by 64 at a time through the kernel for few rows."""
    ops = _ops()
    M, N, K = 70, 3, 0x7f000000 // 1024 + 8
    g = torch.Generator(device="cuda").manual_seed(0)
    a, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda")
    a1 = _rand(M, N)
    got = ops.gemm_f32(a, w, add1=a1)
    want = a1.double()
    for k in range(0, K, 1 << 18):
        want = want + a[:, k:k + (1 << 18)].double() @ w[:, k:k + (1 << 18)].double().T.contiguous()
    assert (got.double() - want).abs().max().item() <= 8 * 2.0 ** -24 * K  # sqrt(K) eps times the root of a sum of K squares
    assert torch.equal(ops.gemm_f32(a[65:].contiguous(), w, add1=a1[65:].contiguous()), got[65:])


@pytest.mark.parametrize("way", [(0, 0, 0, 1), (2, 1, 64, 1), (4, 4, 64, 1), (2, 2, 0, 7), (4, 3, 0, 3)])
def test_products_of_values_without_parts(way):
    """Infinite and undefined values, values that round to an infinite bfloat16, overflow, tiny and huge rows: what 32-bit
    arithmetic says of them, and no change to any other row."""
    ops = _ops()
    M, N, K = 60, 300, 1040
    a, w = _rand(M, K), _rand(N, K, seed=1)
    plain = ops.gemm_f32(a, w)
    b = a.clone()
    b[3, 5], b[7, 9], b[9, 100], b[11, 3] = math.inf, math.nan, 3.4e38, -math.inf
    b[9, :100] *= 1e-10  # the large value alone decides the row, and stays in range where |w| < 1
    b[9, 101:] *= 1e-10
    b[13] *= 1e-30
    b[14] *= 1e34
    b[15] = 3e38 * torch.sign(w[4])  # overflows in column 4, whose products are all positive
    v = w.clone()
    v[20, 3] = 0.0
    fp, fq, whole, share = way
    if fp:
        tiles = -(-N // (64 * fp)) * -(-M // (32 * fq))
        whole = min(whole, tiles)
    got = _product_as(ops, b, v, fp, fq, whole, share)
    want = b.double() @ v.double().T
    row = got[3]
    assert torch.equal(row, torch.where(v[:, 5] > 0, math.inf, -math.inf))
    assert torch.isnan(got[7]).all()
    small = v[:, 100].abs() < 0.99
    torch.testing.assert_close(got[9][small].double(), want[9][small], rtol=1e-5, atol=0.0)
    assert torch.isinf(got[9][v[:, 100].abs() > 1.01]).all()
    other = torch.arange(N, device="cuda") != 20
    assert torch.equal(got[11][other], torch.where(v[other, 3] > 0, -math.inf, math.inf)) and torch.isnan(got[11][20])
    for r in (13, 14):
        scale = (b[r].double() ** 2).sum().sqrt() * (v.double() ** 2).sum(1).sqrt()
        assert ((got[r].double() - want[r]).abs() <= 8 * 2.0 ** -24 * math.sqrt(K) * scale).all()
    assert got[15, 4] == math.inf
    alone = ops.gemm_f32(b[:16].contiguous(), v)  # the kernel for up to sixteen rows
    assert torch.equal(alone.nan_to_num(7.0), got[:16].nan_to_num(7.0))
    same = [r for r in range(M) if r not in (3, 7, 9, 11, 13, 14, 15)]
    assert torch.equal(got[same][:, other], plain[same][:, other])


def _as_way(M, N, way):
    fp, fq, whole, share = way
    return (fp, fq, min(whole, -(-N // (64 * fp)) * -(-M // (32 * fq))) if fp else whole, share)


# down to the smallest 32-bit value, whose parts as bfloat16 exist only beside a factor
@pytest.mark.parametrize("way", [(0, 0, 0, 1), (2, 1, 64, 1), (4, 4, 64, 1), (2, 2, 0, 7), (4, 3, 0, 3)])
@pytest.mark.parametrize("side", ["a", "w"])
def test_products_of_small_values(way, side):
    """Rows of tiny values, of either operand, against large ones: every result relative to its own products."""
    ops = _ops()
    M, N, K = 60, 300, 1040
    small, large = _rand(M if side == "a" else N, K), _rand(N if side == "a" else M, K, seed=1) * 1e30
    powers = [-20, -30, -32, -33, -34, -35, -36, -37, -38, -40, -44]
    small[:len(powers)] = (small[:len(powers)].double() * 10.0 ** torch.tensor(powers, device="cuda").double()[:, None]).float()
    small[20, ::2] *= 1e-36  # beside others
    a, w = (small, large) if side == "a" else (large, small)
    got = _product_as(ops, a, w, *_as_way(M, N, way))
    want = a.double() @ w.double().T
    scale = ((a.double() ** 2) @ (w.double() ** 2).T).sqrt()
    assert ((got.double() - want).abs() <= 8 * 2.0 ** -24 * math.sqrt(K) * scale).all()
    few = ops.gemm_f32(a[:16].contiguous(), w)
    assert torch.equal(few, got[:16])


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 8, 16])
@pytest.mark.parametrize("M", [1, 16, 60, 200])
def test_short_products(M, K):
    """Rows of a few elements: one product is that of 32-bit arithmetic, and several are off by no more than its chain of
    roundings, each under 2^-23 of what has been summed."""
    ops = _ops()
    a, w = _rand(M, K), _rand(300, K, seed=1)
    got = ops.gemm_f32(a, w)
    if K == 1:
        assert torch.equal(got, a * w[:, 0])
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    assert ((got.double() - want).abs() <= K * 2.0 ** -23 * size).all()
    for way in ((0, 0, 0, 1), (2, 1, 64, 1), (4, 4, 0, 1)):
        assert torch.equal(_product_as(ops, a, w, *_as_way(M, 300, way)), got)


def _attention_case(nh, nkv, d, starts, news, window=0, chunk=0, sink=False, slopes=None, spoil=False):
    """(queries, pools, table, token arrays, 64-bit result); pages hold NaN where nothing was written."""
    g = torch.Generator().manual_seed(nh * 100 + d)
    lens = [s + n for s, n in zip(starts, news)]
    pages = [(n + 63) // 64 for n in lens]
    k_pool = torch.full((sum(pages) + 1, nkv, 64, d), float("nan"))
    v_pool = torch.full((sum(pages) + 1, nkv, d, 64), float("nan"))
    table = torch.zeros((len(lens), max(pages)), dtype=torch.int32)
    order = torch.randperm(sum(pages), generator=g).tolist()
    qs, outs = [], []
    sinks = torch.randn(nh, generator=g) if sink else None
    for i, (s0, n, L) in enumerate(zip(starts, news, lens)):
        k, v, q = (torch.randn(m, h, d, generator=g) for m, h in ((L, nkv), (L, nkv), (n, nh)))
        for p in range(pages[i]):
            page = order.pop()
            table[i, p] = page
            m = min(64, L - 64 * p)
            k_pool[page, :, :m] = k[64 * p:64 * p + m].transpose(0, 1)
            v_pool[page, :, :, :m] = v[64 * p:64 * p + m].permute(1, 2, 0)
        qs.append(q)
        j = torch.arange(L)[None, :]
        t = torch.arange(s0, L)[:, None]
        seen = j <= t
        if window:
            seen &= j > t - window
        if chunk:
            seen &= j >= t // chunk * chunk
        o = torch.empty(n, nh, d, dtype=torch.float64)
        for h in range(nh):
            sc = q[:, h].double() @ k[:, h * nkv // nh].double().T * d ** -0.5
            if slopes is not None:
                sc = sc + slopes[h].double() * j * d ** -0.5
            sc = sc.masked_fill(~seen, float("-inf"))
            if sink:
                sc = torch.cat([sc, sinks[h].double().expand(n, 1)], 1)
            o[:, h] = torch.softmax(sc, -1)[:, :L] @ v[:, h * nkv // nh].double()
        outs.append(o.reshape(n, nh * d))
    seq = torch.tensor([i for i, n in enumerate(news) for _ in range(n)], dtype=torch.int32).cuda()
    pos = torch.tensor([s + j for s, n in zip(starts, news) for j in range(n)], dtype=torch.int32).cuda()
    args = (torch.cat(qs).cuda(), k_pool.cuda(), v_pool.cuda(), table.cuda(), seq, pos, None if slopes is None else slopes.cuda(), d ** -0.5)
    kw = dict(window=window, chunk=chunk, sink=None if sinks is None else sinks.cuda(), alibi_exact=True)
    return args, kw, torch.cat(outs)


@pytest.mark.parametrize("nh,nkv,d", [(71, 1, 64), (4, 2, 16), (6, 6, 24), (3, 1, 4), (5, 5, 80), (8, 2, 128), (4, 1, 256), (2, 2, 100), (7, 1, 40)])
@pytest.mark.parametrize("how", ["plain", "window", "chunk", "sink", "slopes"])
def test_attention(nh, nkv, d, how):
    """Prompts, single tokens and continuations of several sequences in one launch, against 64 bits, and one token after the
    other through the kernel for single tokens: the same bits."""
    ops = _ops()
    more = {"window": dict(window=70), "chunk": dict(chunk=96), "sink": dict(sink=True),
            "slopes": dict(slopes=-torch.rand(nh, generator=torch.Generator().manual_seed(3)))}.get(how, {})
    args, kw, want = _attention_case(nh, nkv, d, [0, 63, 700, 0, 127, 64], [70, 1, 5, 1, 2, 200], **more)
    got = ops.attn_generic(*args, **kw)
    assert (got.double().cpu() - want).abs().max().item() <= 2e-5 * max(1.0, want.abs().max().item())
    q, kp, vp, table, seq, pos, slopes, scale = args
    one = ops.attn_generic(*args, **kw, one_each=True)
    assert torch.equal(one, got)
    pick = [0, 69, 70, 75, len(seq) - 1]  # rows of several sequences, each alone
    for r in pick:
        alone = ops.attn_generic(q[r:r + 1].contiguous(), kp, vp, table, seq[r:r + 1].contiguous(), pos[r:r + 1].contiguous(), slopes, scale, **kw)
        assert torch.equal(alone[0], got[r])
    big = torch.full((len(seq), nh * d + 3), 7.0, device="cuda")
    ops.attn_generic(*args, **kw, into=(big[:, 1:1 + nh * d], d, 2.0))
    assert torch.equal(big[:, 1:1 + nh * d], got * 2.0) and bool((big[:, 0] == 7.0).all()) and bool((big[:, -2:] == 7.0).all())


@pytest.mark.parametrize("nh,nkv,d", [(4, 1, 64), (3, 3, 24)])
@pytest.mark.parametrize("window", [0, 5])
@pytest.mark.parametrize("key", [True, False])
def test_attention_hides_values_that_a_token_does_not_see(nh, nkv, d, window, key):
    """An infinite value, and with ``key`` an undefined key, of one token changes no bit of a token that does not see it: earlier
    ones, later ones behind the window, another sequence's; in one launch and token by token.  Whoever sees it shows it."""
    ops = _ops()
    args, kw, _ = _attention_case(nh, nkv, d, [0, 0], [50, 30], window=window)
    got = ops.attn_generic(*args, **kw)
    q, kp, vp, table, *rest = args
    kp, vp = kp.clone(), vp.clone()
    vp[table[0, 0].item(), :, :, 40] = float("inf")
    if key:
        kp[table[0, 0].item(), :, 40] = float("nan")
    sees = slice(40, 40 + window if window else 50)
    for one_each in (False, True):
        bad = ops.attn_generic(q, kp, vp, table, *rest, **kw, one_each=one_each)
        assert torch.equal(bad[:40], got[:40]) and torch.equal(bad[sees.stop:], got[sees.stop:])
        assert bool(torch.isnan(bad[sees]).all() if key else (bad[sees] == float("inf")).all())


def _step(runs, nh, nkv, d, seed=0):
    """(attn_generic's arguments, the step's context) for sequences of (cached, new) tokens with random keys and values."""
    from types import SimpleNamespace

    g = torch.Generator(device="cuda").manual_seed(seed)
    starts, news = [a for a, _ in runs], [b for _, b in runs]
    pages = [(a + b + 63) // 64 for a, b in runs]
    order = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(seed)).int()
    table, at = torch.zeros((len(runs), max(pages)), dtype=torch.int32), 0
    for i, n in enumerate(pages):
        table[i, :n] = order[at:at + n]
        at += n
    new = lambda *shape: torch.randn(*shape, generator=g, device="cuda")
    ints = lambda v: torch.tensor(v, dtype=torch.int32).cuda()
    cu = [0]
    for n in news:
        cu.append(cu[-1] + n)
    ctx = SimpleNamespace(is_decode=all(n == 1 for n in news), n_seqs=len(runs), new_tokens=news, starts=starts, cu_tokens=ints(cu),
                          max_len=max(a + b for a, b in runs), extras={})
    args = (new(cu[-1], nh, d), new(sum(pages), nkv, 64, d), new(sum(pages), nkv, d, 64), table.cuda(),
            ints([i for i, n in enumerate(news) for _ in range(n)]), ints([a + j for a, n in runs for j in range(n)]), None, d ** -0.5)
    return args, ctx


@pytest.mark.parametrize("nh,nkv,d", [(71, 1, 64), (16, 16, 64), (3, 1, 100), (4, 2, 256), (6, 2, 16)])
@pytest.mark.parametrize("runs", [
    [(600, 1)] * 70 + [(0, 1200)] + [(64, 1)] * 3,      # single tokens beside a prompt, more than 64 sequences
    [(500, 3), (0, 1), (130, 40), (0, 129)],            # a few tokens behind many
    [(0, 33)] * 130 + [(0, 700)],                       # short prompts, more than 128 of them
    [(0, 1)] * 5 + [(63, 1), (64, 1), (900, 1)],        # one token each
    [(40 * i, 1) for i in range(300)],                  # so many of them that a wave takes each
])
def test_attention_of_steps(nh, nkv, d, runs):
    """A step's launches, however its sequences are shared out, against every token by itself: the same bits, with and without a
    window."""
    ops = _ops()
    args, ctx = _step(runs, nh, nkv, d)
    for kw in ({}, {"window": 70}):
        assert torch.equal(ops.attn_generic(*args, **kw, ctx=ctx), ops.attn_generic(*args, **kw))


def test_attention_of_steps_takes_both_kernels():
    """A mixed step shares the single tokens' pages out and not the prompt's, and a large batch of prompts has
    two tiles a wave."""
    ops = _ops()
    for runs, shared, prompts, tiles in (([(600, 1)] * 40 + [(0, 1200)], True, True, 2), ([(0, 256)] * 8, False, True, 2),
                                         ([(0, 1)] * 300, False, True, 1), ([(900, 3), (70, 1)], True, False, 1)):
        args, ctx = _step(runs, 71, 1, 64)
        assert torch.equal(ops.attn_generic(*args, ctx=ctx), ops.attn_generic(*args))
        plan = next(iter(ctx.extras.values()))
        assert (plan.shared_tiles > 0, plan.prompt_waves > 0, plan.wave_tiles) == (shared, prompts, tiles)


def test_a_prompt_beside_single_tokens_costs_what_the_two_cost():
    """32 single tokens behind 1,000 keys and a prompt of 64 tokens in one step, 16 heads on as many KV heads: no more than a few
    times the two steps apart (a wave that walks one sequence after the other for its sixteen heads took a hundred times as long)."""
    ops = _ops()

    def us(runs):
        args, ctx = _step(runs, 16, 16, 64)
        ctx.seq_start = torch.tensor(ctx.starts, dtype=torch.int32).cuda()
        ctx.block_tables, ctx.token_seq, ctx.token_pos, best = None, args[4], args[5], float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(10):
                ops.attention(*args[:4], ctx, None, args[7])
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 100)
        return best

    apart = us([(1000, 1)] * 32) + us([(0, 64)])
    assert us([(1000, 1)] * 32 + [(0, 64)]) <= 4 * apart + 50


@pytest.mark.parametrize("M,N1,K1,N2,K2", [(1, 4672, 4544, 18176, 4544), (16, 4544, 4544, 4544, 18176), (7, 36, 64, 1000, 68),
                                           (2, 3, 1024, 4100, 8), (16, 8193, 260, 8193, 28), (5, 2064, 2048, 2064, 1028)])
def test_two_products_in_one_launch_are_the_products_on_their_own(M, N1, K1, N2, K2):
    """Bit by bit, with biases, activations and the sum of the two: workgroups with rows of one matrix alone, waves without a segment of
    one K, one tile of sixteen rows and two."""
    ops = _ops()
    g = torch.Generator(device="cuda").manual_seed(M + N1 + K2)
    draw = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    a1, w1, b1, a2, w2, b2 = draw(M, K1), draw(N1, K1), draw(N1), draw(M, K2), draw(N2, K2), draw(N2)
    assert ops.gemm_f32_pair_ok(a1, w1, a2, w2)
    got = ops.gemm_f32_pair(a1, w1, a2, w2, b1, None, b2, "gelu")
    assert torch.equal(got[0], ops.gemm_f32(a1, w1, b1))
    assert torch.equal(got[1], ops.gemm_f32(a2, w2, b2, "gelu"))
    if N1 == N2:
        x = draw(M, N2)
        first = ops.gemm_f32(a1, w1, b1)
        for bias, add in ((b2, x), (None, None)):
            assert torch.equal(ops.gemm_f32_pair_sum(a1, w1, a2, w2, b1, bias, add), ops.gemm_f32(a2, w2, bias, None, first, add))
        big = a1.clone()
        big[0, 3] = float("inf")  # a sum that is formed on the 32-bit instruction
        want = ops.gemm_f32(a2, w2, None, None, ops.gemm_f32(big, w1), None)
        assert torch.equal(torch.nan_to_num(ops.gemm_f32_pair_sum(big, w1, a2, w2)), torch.nan_to_num(want))


def test_pairs_that_have_no_launch():
    w = lambda n, k: torch.empty((n, k), device="cuda")
    ok = _ops().gemm_f32_pair_ok
    assert not ok(w(17, 2048), w(64, 2048), w(17, 2048), w(64, 2048))  # more rows than the rings take
    assert not ok(w(1, 6), w(64, 6), w(1, 8), w(64, 8))  # rows that are no multiple of sixteen bytes
    assert not ok(w(1, 64), w(64, 64), w(2, 64), w(64, 64))
    assert not ok(w(1, 64), w(64, 64), w(1, 64), w(60, 64), add_first=True)
    assert not ok(w(1, 8192), w(32768, 8192), w(1, 8192), w(64, 8192))  # a matrix that goes by tiles
    assert not ok(w(1, 64).bfloat16(), w(64, 64).bfloat16(), w(1, 64).bfloat16(), w(64, 64).bfloat16())
