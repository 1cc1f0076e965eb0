"""Decode attention over contexts of 193 to 1,024 keys, 512 on average: four waves of a workgroup share a context."""
import pytest
import torch
from types import SimpleNamespace

from pytorch_transformers_amd import ops, tuning

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(bool(ops.ATTN_FORCE_SPLIT or ops.ATTN_FORCE_TILES), reason="the cut is set by PTA_ATTN_SPLIT or PTA_ATTN_TILES")]


@pytest.mark.parametrize("nh,nkv,d", [(13, 13, 80), (71, 1, 64), (4, 2, 16), (64, 8, 64)])
@pytest.mark.parametrize("lens", [[193], [1024, 1, 31, 32, 33], [200, 511, 64, 65, 127, 128, 129, 300], [260] * 24 + [200] * 8])
def test_against_plain_attention(nh, nkv, d, lens):
    """Contexts that give a wave no block, a part of one or several; weights and results are rounded to bfloat16, 2^-8 of the
    largest value each."""
    g = torch.Generator().manual_seed(len(lens) + d)
    n, width = len(lens), 16
    pages = n * width
    k_pool, v_pool = torch.full((pages, nkv, 64, d), float("nan")), torch.full((pages, nkv, d, 64), float("nan"))
    table = torch.randperm(pages, generator=g).view(n, width).int()
    q = torch.randn(n, nh, d, generator=g).bfloat16()
    want = []
    for i, L in enumerate(lens):
        k, v = torch.randn(L, nkv, d, generator=g).bfloat16(), torch.randn(L, nkv, d, generator=g).bfloat16()
        for p in range((L + 63) // 64):
            m = min(64, L - 64 * p)
            k_pool[table[i, p], :, :m] = k[64 * p:64 * p + m].float().transpose(0, 1)
            v_pool[table[i, p], :, :, :m] = v[64 * p:64 * p + m].float().permute(1, 2, 0)
        kk, vv = (t.double().repeat_interleave(nh // nkv, 1) for t in (k, v))
        a = torch.softmax((q[i].double()[None] * kk).sum(-1).t() * d ** -0.5, -1)
        want.append((a.t()[:, :, None] * vv).sum(0).reshape(-1))
    want = torch.stack(want)
    pos = torch.tensor([L - 1 for L in lens], dtype=torch.int32).cuda()
    mean = min(1024, -(-sum(lens) // n // 512) * 512 or 512)
    ctx = SimpleNamespace(is_decode=True, n_seqs=n, max_len=max(lens), mean_len=mean, new_tokens=[1] * n, token_pos=pos, seq_start=pos,
                          cu_tokens=torch.arange(n + 1, dtype=torch.int32).cuda(), token_seq=torch.arange(n, dtype=torch.int32).cuda())
    cut = tuning.several_waves_cut(n, nh, nkv, d, max(lens), mean)
    groups = (1 << (n - 1).bit_length()) * nkv * ((nh // nkv + 15) // 16)
    assert cut == ((1, 1024, 4) if groups <= 320 and ops.load_library().pta_attn_decode_waves_ok(d, 1, 4) else None)
    got = ops.attention(q.cuda(), k_pool.bfloat16().cuda(), v_pool.bfloat16().cuda(), table.cuda(), ctx, None, d ** -0.5)
    assert (got.double().cpu() - want).abs().max().item() <= 2 ** -7 * want.abs().max().item()


def test_where_it_applies():
    assert tuning.several_waves_cut(5, 13, 13, 80, 325, 512) == (1, 1024, 4)
    assert tuning.several_waves_cut(5, 13, 13, 80, 325, 300) == tuning.several_waves_cut(8, 13, 13, 80, 1024, 512)  # a step's bucket
    assert tuning.several_waves_cut(5, 13, 13, 80, 1025, 512) is None and tuning.several_waves_cut(5, 13, 13, 80, 900, 600) is None
    assert tuning.several_waves_cut(64, 128, 8, 64, 300, 300) is None and tuning.several_waves_cut(8, 32, 8, 128, 300, 300) is None
    assert tuning.several_waves_cut(32, 32, 8, 128, 300, 300) == (1, 1024, 4)
    key = ops.decode_key(5, 13, 13, 80, 325, 300)
    ops.set_decode_plan(key, (1, 128, 1))  # a timed cut goes before the rule
    try:
        assert tuning.several_waves_cut(5, 13, 13, 80, 325, 300) is None and ops.decode_plan(5, 13, 13, 80, 325, 300) == (1, 128, 1)
    finally:
        ops.set_decode_plan(key, None)


@pytest.mark.parametrize("n,nh,nkv,d,max_len,mean", [(5, 13, 13, 80, 325, 300), (64, 71, 1, 64, 500, 400), (64, 71, 1, 64, 1100, 1000), (8, 32, 8, 128, 300, 300)])
def test_what_is_measured_first_is_what_runs_untuned(monkeypatch, n, nh, nkv, d, max_len, mean):
    """``CausalLM.tune`` keeps no entry where the first candidate was the fastest: it has to be the cut of the launch without one."""
    width = (max_len + 63) // 64
    pool = torch.zeros(n * width, nkv, 64, d, dtype=torch.bfloat16, device="cuda")
    table = torch.arange(n * width, dtype=torch.int32, device="cuda").view(n, width)
    pos = torch.full((n,), max_len - 1, dtype=torch.int32, device="cuda")
    ctx = SimpleNamespace(is_decode=True, n_seqs=n, max_len=max_len, mean_len=mean, new_tokens=[1] * n, token_pos=pos, seq_start=pos,
                          cu_tokens=torch.arange(n + 1, dtype=torch.int32).cuda(), token_seq=torch.arange(n, dtype=torch.int32).cuda())
    ran, attn = [], ops.attn_mfma
    monkeypatch.setattr(ops, "attn_mfma", lambda *a, **k: (ran.append(k), attn(*a, **k))[1])
    launch = lambda: (ops.attention(torch.zeros(n, nh, d, dtype=torch.bfloat16, device="cuda"), pool, pool.view(-1, nkv, d, 64), table, ctx, None, 1.0),
                      ran.pop())[1]
    key = ops.decode_key(n, nh, nkv, d, max_len, mean)
    ops.set_decode_plan(key, None)
    cuts, untuned = ops.decode_plan_candidates(key), launch()
    assert len(set(cuts)) == len(cuts) and (tuning.several_waves_cut(n, nh, nkv, d, max_len, mean) or ops.decode_plan(n, nh, nkv, d, max_len, mean)) == cuts[0]
    try:
        ops.set_decode_plan(key, cuts[0])
        assert launch() == untuned
        ops.set_decode_plan(key, cuts[1])
        assert launch() != untuned
    finally:
        ops.set_decode_plan(key, None)
    assert launch() == untuned
