"""A decode step's attention in the launch of the two products behind it: the bits of the launches on their own."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


def _step(M, nh, nkv, longest, seed, d=64):
    """Queries, pages and tables of M sequences of 1 to ``longest`` keys."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    lens = [longest] + [int(n) for n in torch.randint(1, longest + 1, (M - 1,), generator=torch.Generator().manual_seed(seed))]
    width = (longest + 63) // 64
    pages = torch.randperm(M * width, generator=torch.Generator().manual_seed(seed)).to(torch.int32).cuda().view(M, width)
    draw = lambda *shape: torch.randn(shape, generator=g, device="cuda").bfloat16()
    k_pool, v_pool = draw(M * width, nkv, 64, d), draw(M * width, nkv, d, 64)
    for m, n in enumerate(lens):  # what lies past a sequence's end is never seen
        if n % 64:
            k_pool[pages[m, (n - 1) // 64].long(), :, n % 64:] = float("nan")
            v_pool[pages[m, (n - 1) // 64].long(), :, :, n % 64:] = float("nan")
    ctx = types.SimpleNamespace(cu_tokens=torch.arange(M + 1, dtype=torch.int32, device="cuda"), n_seqs=M, max_len=longest, mean_len=longest,
                                seq_start=torch.tensor([n - 1 for n in lens], dtype=torch.int32, device="cuda"), is_decode=True, new_tokens=[1] * M, extras={})
    return draw(M, nh, d), k_pool, v_pool, pages, ctx, draw


@pytest.mark.parametrize("owners,waves", [(-1, 1), (0, 1), (-1, 4), (0, 4), (3, 4)])
@pytest.mark.parametrize("M,nh,nkv,N,K1,longest", [(1, 71, 1, 4544, 18176, 60), (8, 71, 1, 4544, 18176, 700), (16, 32, 8, 2048, 8192, 129),
                                                   (17, 17, 1, 1096, 4352, 33), (33, 71, 1, 4544, 18176, 300), (64, 16, 2, 2056, 4096, 1), (48, 128, 8, 8192, 32768, 200)])
def test_attention_rides_with_the_products(M, nh, nkv, N, K1, longest, owners, waves):
    """Every height of the tiles, walks from a stage of their own and from the start, groups of heads that fill no tile, and with
    attention done by its own workgroups, by some of them, and by those that wait for it alone."""
    from pytorch_transformers_amd import ops

    q, k_pool, v_pool, table, ctx, draw = _step(M, nh, nkv, longest, seed=M + nh)
    x1, w1, w2 = draw(M, K1), draw(N, K1) * 0.05, draw(N, nh * 64) * 0.05
    late = ops.LateAttention(q, k_pool, v_pool, table, ctx, None, 0.125, waves=waves)
    assert ops.gemm_splitk_pair_attn_ok(x1, w1, late, w2)
    want = ops.attn_mfma(q, k_pool, v_pool, table, ctx.cu_tokens, ctx.seq_start, None, 0.125, max_new=1, decode_tiles=1, decode_waves=waves)
    assert torch.isfinite(want.float()).all()
    parts = ops.gemm_splitk_pair_partial(x1, w1, want, w2)
    for _ in range(3):  # (marks of their own each time)
        late.out.fill_(float("nan"))
        got = ops.gemm_splitk_pair_attn(x1, w1, late, w2, owners=owners)
        assert torch.equal(late.out, want)
        assert torch.equal(got[0], parts[0]) and torch.equal(got[1], parts[1])


def test_a_bias_on_the_scores_and_a_sink():
    from pytorch_transformers_amd import ops

    q, k_pool, v_pool, table, ctx, draw = _step(5, 32, 8, 150, seed=3)
    slopes, sink = torch.rand(32, device="cuda") * 0.1, torch.randn(32, device="cuda")
    x1, w1, w2 = draw(5, 8192), draw(2048, 8192), draw(2048, 2048)
    for how in (dict(sink=sink), dict(alibi_exact=True, bias_of="distance", bias_scale=1.0), dict(alibi_exact=False, sink=sink)):
        bias = slopes if "alibi_exact" in how else None
        late = ops.LateAttention(q, k_pool, v_pool, table, ctx, bias, 0.125, **how)
        want = ops.attn_mfma(q, k_pool, v_pool, table, ctx.cu_tokens, ctx.seq_start, bias, 0.125, max_new=1, decode_tiles=1, decode_waves=4, **how)
        ops.gemm_splitk_pair_attn(x1, w1, late, w2)
        assert torch.equal(late.out, want)


def test_captured_launches_are_replayed():
    """The marks are cleared by the capture itself: replays with the program's own work between them give the same."""
    from pytorch_transformers_amd import ops

    q, k_pool, v_pool, table, ctx, draw = _step(8, 71, 1, 100, seed=9)
    x1, w1, w2 = draw(8, 18176), draw(4544, 18176), draw(4544, 4544)
    want = ops.attn_mfma(q, k_pool, v_pool, table, ctx.cu_tokens, ctx.seq_start, None, 0.125, max_new=1, decode_tiles=1, decode_waves=4)
    parts = ops.gemm_splitk_pair_partial(x1, w1, want, w2)
    graph, stream, outs = torch.cuda.CUDAGraph(), torch.cuda.Stream(), []
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        graph.capture_begin()
        for _ in range(40):  # more than are cleared at a time
            late = ops.LateAttention(q, k_pool, v_pool, table, ctx, None, 0.125)
            outs.append((late.out,) + ops.gemm_splitk_pair_attn(x1, w1, late, w2))
        graph.capture_end()
    for _ in range(4):
        for out in outs:
            out[0].fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        q.sum().item()
        for out, a, b in outs:
            assert torch.equal(out, want) and torch.equal(a, parts[0]) and torch.equal(b, parts[1])
    ctx.extras.clear()


def test_a_decode_step_takes_the_launch(monkeypatch):
    """Steps of a parallel model with heads of 64 over short contexts, directly and as replays, against the launches on their own."""
    from pytorch_transformers_amd import AutoModelForCausalLM, FalconConfig, ops, tuning

    cfg = FalconConfig(num_hidden_layers=3, hidden_size=1024, num_attention_heads=16, multi_query=True, new_decoder_architecture=False, parallel_attn=True,
                       vocab_size=512, ffn_hidden_size=16384, alibi=False, bias=False)
    model = AutoModelForCausalLM.from_config(cfg, seed=0, std=0.05, dtype="bfloat16", device="cuda:0")
    calls = []
    launch = ops.gemm_splitk_pair_attn
    monkeypatch.setattr(ops, "gemm_splitk_pair_attn", lambda *a, **k: calls.append(1) or launch(*a, **k))

    def logits(n):
        cache = model.new_cache(1024, max_slots=n)
        slots = [cache.alloc() for _ in range(n)]
        model.step(cache, slots, [[1 + i] * (3 + i) for i in range(n)], "last")
        return torch.stack([model.step(cache, slots, [[7 + i + j] for i in range(n)], "last") for j in range(4)])

    for n in (1, 5):
        got = logits(n)
        assert len(calls) == 6  # three layers directly, and three captured
        monkeypatch.setattr(tuning, "late_waves", lambda *a: 0)
        want = logits(n)
        assert len(calls) == 6
        monkeypatch.undo()
        monkeypatch.setattr(ops, "gemm_splitk_pair_attn", lambda *a, **k: calls.append(1) or launch(*a, **k))
        calls.clear()
        model._captured_shapes.clear()
        assert torch.equal(got, want)
