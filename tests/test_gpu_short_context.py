"""Decode attention over short contexts, which one wave per sequence and group of heads walks whole, around the length at which
that ends, against 64 bits; and captured decode steps across that length."""
import math
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,d", [(71, 1, 64), (13, 13, 80), (16, 8, 128), (4, 1, 256), (2, 2, 16)])
@pytest.mark.parametrize("longest", [1, 64, 65, 191, 192, 193])
def test_decode_attention(nh, nkv, d, longest):
    from pytorch_transformers_amd import ops, tuning

    g = torch.Generator().manual_seed(longest)
    lens = [longest, max(1, longest // 2), 1]
    n, width = len(lens), tuning.context_bound(longest) // 64
    k_pool = torch.full((n * width + 1, nkv, 64, d), float("nan"))
    v_pool = torch.zeros((n * width + 1, nkv, d, 64))
    table = torch.randperm(n * width, generator=g).view(n, width).int()
    want, q = [], torch.randn(n, nh, d, generator=g).bfloat16()
    for i, L in enumerate(lens):
        k, v = torch.randn(L, nkv, d, generator=g).bfloat16(), torch.randn(L, nkv, d, generator=g).bfloat16()
        for j in range(L):
            k_pool[table[i, j // 64], :, j % 64] = k[j].float()
            v_pool[table[i, j // 64], :, :, j % 64] = v[j].float()
        kk, vv = (t.double().repeat_interleave(nh // nkv, 1) for t in (k, v))
        a = torch.softmax(torch.einsum("hd,jhd->hj", q[i].double(), kk) * d ** -0.5, -1)
        want.append(torch.einsum("hj,jhd->hd", a, vv).reshape(-1))
    pos = torch.tensor([L - 1 for L in lens], dtype=torch.int32).cuda()
    ctx = SimpleNamespace(is_decode=True, n_seqs=n, max_len=longest, mean_len=longest, new_tokens=[1] * n, token_pos=pos, seq_start=pos,
                          cu_tokens=torch.arange(n + 1, dtype=torch.int32).cuda(), token_seq=torch.arange(n, dtype=torch.int32).cuda())
    got = ops.attention(q.cuda(), k_pool.bfloat16().cuda(), v_pool.bfloat16().cuda(), table.cuda(), ctx, None, d ** -0.5)
    want = torch.stack(want)
    # weights and results are rounded to bfloat16: 2^-8 of the largest value each
    assert (got.double().cpu() - want).abs().max().item() <= 2 ** -7 * want.abs().max().item()
    assert (tuning.short_cut(longest) is None) == (longest > 192)


def test_captured_steps_across_the_bound():
    """Greedy tokens of one sequence from 180 to 205 tokens: captured steps against direct ones, bit for bit."""
    from pytorch_transformers_amd import AutoModelForCausalLM, FalconConfig

    cfg = FalconConfig(num_hidden_layers=2, hidden_size=128, num_attention_heads=4, num_kv_heads=2, new_decoder_architecture=True,
                       vocab_size=500, ffn_hidden_size=256, alibi=False, bias=False)
    model = AutoModelForCausalLM.from_config(cfg, seed=0, std=0.2, dtype="bfloat16", device="cuda:0")
    g = torch.Generator().manual_seed(1)
    prompts = [torch.randint(0, 500, (n,), generator=g).tolist() for n in (180, 20)]
    feed = torch.randint(0, 500, (25, 2), generator=g).tolist()
    runs = []
    for graphs in (True, False):
        model.use_graphs = graphs
        cache = model.new_cache(1024, max_slots=2)
        slots = [cache.alloc(), cache.alloc()]
        rows = [model.step(cache, slots, prompts, "last")]
        rows += [model.step(cache, slots, [[t] for t in ts], "last") for ts in feed]
        runs.append(torch.stack(rows))
    assert torch.equal(runs[0], runs[1]) and math.isfinite(float(runs[0].sum()))
