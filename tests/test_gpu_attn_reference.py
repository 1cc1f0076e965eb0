"""The running maximum that attention's exponentials are taken against: every wave's own scores, whichever kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pools(n_pages, nkv, d, g):
    k = torch.randn((n_pages, nkv, 64, d), generator=g).bfloat16()
    v = torch.randn((n_pages, nkv, d, 64), generator=g).bfloat16()
    return k, v


def _exact(q, k, v, table, lens, scale):
    """[tokens, heads, d] in 64 bits; one token a sequence, or a prompt's tokens (new of them, the sequence's last)."""
    out, at = [], 0
    for s, (n, new) in enumerate(lens):
        nkv, d = k.shape[1], k.shape[3]
        K = torch.cat([k[p] for p in table[s]], 1)[:, :n].double()                        # [nkv, n, d]
        V = torch.cat([v[p].transpose(1, 2) for p in table[s]], 1)[:, :n].double()
        g = q.shape[1] // nkv
        for t in range(new):
            sees = n - new + t + 1
            row = q[at + t].double().view(nkv, g, d)
            w = torch.softmax(torch.bmm(row, K[:, :sees].transpose(1, 2).contiguous()) * scale, -1)
            out.append(torch.bmm(w, V[:, :sees].contiguous()).reshape(-1, d))
        at += new
    return torch.stack(out)


@pytest.mark.parametrize("heads,kv,d", [(49, 1, 64), (64, 1, 64), (71, 1, 64), (80, 1, 64), (100, 1, 64), (71, 1, 128), (128, 1, 128), (16, 2, 64), (8, 2, 80)])
@pytest.mark.parametrize("spread", [1.0, 40.0])
def test_scores_of_any_size(heads, kv, d, spread):
    """Scores that lie hundreds of units apart from block to block (``spread`` 40) are weighed against a maximum that was read when it was there: one
    that is missed leaves infinities, and one that is something else another result each time.  Decode launches of every kind and prompts."""
    from pytorch_transformers_amd import ops

    g = torch.Generator().manual_seed(heads + d)
    k, v = _pools(12, kv, d, g)
    table = [[3, 0, 5, 1, 8, 9], [7, 2, 4, 6, 10, 11]]
    i32 = lambda t: torch.tensor(t, dtype=torch.int32).cuda()
    for new in ((1, 1), (90, 30)):
        lens = [(350, new[0]), (171, new[1])]
        q = (torch.randn((sum(new), heads, d), generator=g) * spread).bfloat16()
        want = _exact(q, k, v, table, lens, d ** -0.5)
        ways = [dict()]
        if new[0] == 1:
            ways = [dict(n_splits=1, split_size=512), dict(n_splits=2, split_size=192)]
            if ops.load_library().pta_attn_decode_waves_ok(d, 1, 4):
                ways.append(dict(n_splits=1, split_size=512, decode_tiles=1, decode_waves=4))
            if ops.attn_decode_shared_ok(d, heads // kv):
                ways += [dict(n_splits=n, split_size=384 // n, decode_waves=ops.SHARED_KEYS) for n in (1, 2)]
        args = (q.cuda(), k.cuda(), v.cuda(), i32(table), i32([0, new[0], sum(new)]), i32([n - m for n, m in lens]), None, d ** -0.5)
        for way in ways:
            outs = [ops.attn_mfma(*args, max_new=max(new), **way).view(sum(new), heads, d) for _ in range(4)]
            # weights and results are rounded to bfloat16 (2^-9 each, of values of about one)
            off = float((outs[0].double().cpu() - want).abs().max())
            assert off <= 2.0 ** -6 * float(want.abs().max()), f"{way}: off by {off}"
            assert all(torch.equal(outs[0], o) for o in outs[1:]), f"{way}: not the same bits each time"
