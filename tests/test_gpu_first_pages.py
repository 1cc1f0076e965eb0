"""Decode attention whose waves look their first two pages up before they know the sequence's length: page lists as wide as the
longest sequence needs and no wider, entries behind a sequence's end that name no page."""
import pytest
import torch

from pytorch_transformers_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh,nkv,d", [(3, 3, 80), (8, 1, 64)])
@pytest.mark.parametrize("lens", [[1], [64, 1], [65, 32, 33], [129, 128, 1, 64, 127], [321, 5, 192, 193], [640, 31]])
@pytest.mark.parametrize("size,waves", [(0, 1), (0, 4), (0, 8), (64, 1), (128, 1), (256, 4)])
def test_against_plain_attention(nh, nkv, d, lens, size, waves):
    if waves > 1 and not ops.load_library().pta_attn_decode_waves_ok(d, 1, waves):
        pytest.skip("not built")
    g = torch.Generator().manual_seed(sum(lens) + d)
    n, width = len(lens), (max(lens) + 63) // 64
    pages = sum((L + 63) // 64 for L in lens)
    k_pool, v_pool = torch.full((pages, nkv, 64, d), float("nan")), torch.full((pages, nkv, d, 64), float("nan"))
    table, order, at = torch.full((n, width), -1, dtype=torch.int32), torch.randperm(pages, generator=g).tolist(), 0
    q = torch.randn(n, nh, d, generator=g).bfloat16()
    want = []
    for i, L in enumerate(lens):
        k, v = torch.randn(L, nkv, d, generator=g).bfloat16(), torch.randn(L, nkv, d, generator=g).bfloat16()
        for p in range((L + 63) // 64):
            m = min(64, L - 64 * p)
            table[i, p], at = order[at], at + 1
            k_pool[table[i, p], :, :m] = k[64 * p:64 * p + m].float().transpose(0, 1)
            v_pool[table[i, p], :, :, :m] = v[64 * p:64 * p + m].float().permute(1, 2, 0)
        kk, vv = (t.double().repeat_interleave(nh // nkv, 1) for t in (k, v))
        a = torch.softmax((q[i].double()[None] * kk).sum(-1).t() * d ** -0.5, -1)
        want.append((a.t()[:, :, None] * vv).sum(0).reshape(-1))
    want = torch.stack(want)
    size = size or -(-max(lens) // 64) * 64
    start = torch.tensor([L - 1 for L in lens], dtype=torch.int32).cuda()
    got = ops.attn_mfma(q.cuda(), k_pool.bfloat16().cuda(), v_pool.bfloat16().cuda(), table.cuda(), torch.arange(n + 1, dtype=torch.int32).cuda(),
                        start, None, d ** -0.5, max_new=1, n_splits=-(-max(lens) // size), split_size=size, decode_tiles=1, decode_waves=waves)
    assert (got.double().cpu() - want).abs().max().item() <= 2 ** -7 * want.abs().max().item()  # weights and results: 2^-8 each
