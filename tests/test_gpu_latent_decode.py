"""The decode launches over a cache of latents against 64 bits, at the edges of their tiles: heads beyond sixteen, latents from
one piece of 32 elements to 512, no rotated part, outputs that fill no tile, contexts around a page and a range, ranges of one
page and of several."""
from types import SimpleNamespace

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,dn,dr,R,V", [(16, 128, 64, 512, 128), (1, 32, 0, 32, 16), (17, 64, 32, 96, 40), (40, 256, 64, 192, 100), (3, 96, 128, 512, 33)])
@pytest.mark.parametrize("lens", [[1], [64, 65, 1], [700, 3, 130], [100] * 17, [max(1, 700 - 23 * i) for i in range(33)]])
def test_against_64_bits(H, dn, dr, R, V, lens):
    from pytorch_transformers_amd import ops

    g = torch.Generator().manual_seed(H + dn + len(lens))
    r = lambda *s: torch.randn(*s, generator=g)
    M, D, width = len(lens), R + dr, (max(lens) + 63) // 64
    assert M < 33 or ops.latent_ranges(M, H, max(lens))[0] > 64  # ranges of several pages, which end inside one
    assert ops.latent_decode_ok(torch.empty(M, 1, dtype=torch.bfloat16), H, dn, dr, R, V)
    table = torch.randperm(M * width, generator=g).view(M, width).int()
    pool = torch.full((M * width + 1, 1, 64, D), float("nan"))
    rows = [r(n, D).bfloat16() for n in lens]
    for i, n in enumerate(lens):
        for j in range(n):
            pool[table[i, j // 64], 0, j % 64] = rows[i][j].float()
    q, kt, up_v = r(M, H * (dn + dr)).bfloat16(), (0.1 * r(H, R, dn)).bfloat16(), (0.1 * r(H, V, R)).bfloat16()
    down, w_norm = r(M, D).bfloat16(), 1 + 0.1 * r(R)
    pos = torch.tensor([n - 1 for n in lens], dtype=torch.int32).cuda()
    inv = (10000.0 ** (-torch.arange(dr // 2).float() * 2 / dr)).cuda() if dr else None
    pool = pool.bfloat16().cuda()
    before = pool.clone()
    seq = torch.arange(M, dtype=torch.int32).cuda()
    ref_pool = pool.clone()
    args = (down.cuda(), w_norm.cuda(), 1e-6, inv, 1.0, dr, "interleaved", pos, seq, table.cuda())
    frames = ops.latent_queries(*args, pool, kt.cuda(), H, dn, dr, R, write_cache=True, q=q.cuda())
    plain = ops.latent_prep(*args, ref_pool, H, dn, dr, R, write_cache=True, q=q.cuda())
    # the cache rows and the rotated parts are latent_prep's, bit for bit; the rest is the expansion
    assert torch.equal(torch.nan_to_num(pool.float(), 7.0), torch.nan_to_num(ref_pool.float(), 7.0))
    assert torch.equal(frames[:, :, R:], plain[:, :, R:])
    want = torch.einsum("mhd,hrd->mhr", q.view(M, H, dn + dr)[:, :, :dn].double(), kt.double())
    assert (frames[:, :, :R].double().cpu() - want).abs().max().item() <= 2.0 ** -18 * dn ** 0.5 * want.abs().max().item()
    none = ops.latent_queries(None, None, 1e-6, *args[3:], before, kt.cuda(), H, dn, dr, R, write_cache=False, q=q.cuda())
    assert torch.equal(none, frames)
    ctx = SimpleNamespace(max_len=max(lens), seq_start=pos)
    scale = D ** -0.5
    got = ops.latent_decode(frames, pool, table.cuda(), up_v.cuda(), R, scale, ctx).double().cpu().view(M, H, V)
    for i, n in enumerate(lens):
        keys = torch.stack([pool[table[i, j // 64], 0, j % 64].double().cpu() for j in range(n)])
        a = torch.softmax(frames[i].double().cpu() @ keys.T * scale, -1)
        out = torch.einsum("hr,hvr->hv", a @ keys[:, :R], up_v.double())
        # queries, weights and latents are rounded to bfloat16 on the way: 2^-8 each, times the spread that a score of size s has
        assert (got[i] - out).abs().max().item() <= 2.0 ** -5 * max(out.abs().max().item(), 0.1), f"sequence {i}"
