"""Keys and values of many tokens in their pages: steps whose values go by a launch of their own leave the same bits as the same
tokens in steps small enough to write them where queries and keys are rotated."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nh,nkv,d,layout,rotate", [(4, 2, 64, "grouped", True), (6, 1, 256, "tail", True), (3, 3, 40, "interleaved", False),
                                                    (8, 8, 33, "grouped", False), (4, 4, 128, "grouped", True)])
def test_value_pages(nh, nkv, d, layout, rotate, dtype):
    """Ragged sequences that begin inside pages, head sizes below, at and above a tile of 64 elements and of odd size."""
    from pytorch_transformers_amd import ops

    ops.load_library()
    lens, starts = [1, 63, 9000, 129, 2, 9000], [70, 1, 5, 63, 64, 0]
    M, g = sum(lens), torch.Generator().manual_seed(d)
    pages = [(s + n + 63) // 64 for s, n in zip(starts, lens)]
    table, order = torch.zeros((len(lens), max(pages)), dtype=torch.int32), torch.randperm(sum(pages), generator=g).int()
    for i, n in enumerate(pages):
        table[i, :n] = order[sum(pages[:i]):sum(pages[:i + 1])]
    fused = torch.randn(M, (nh + 2 * nkv) * d, generator=g).to(dtype).cuda()
    bias = torch.randn((nh + 2 * nkv) * d, generator=g).cuda()
    pos = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lens)]).int().cuda()
    seq = torch.cat([torch.full((n,), i) for i, n in enumerate(lens)]).int().cuda()
    freq = (1e4 ** -(torch.arange(0, d, 2) / d)).cuda() if rotate else None
    table = table.cuda()

    def run(step):
        k = torch.zeros((sum(pages), nkv, 64, d), dtype=dtype, device="cuda")
        v = torch.zeros((sum(pages), nkv, d, 64), dtype=dtype, device="cuda")
        q = [ops.qkv_rope_cache(fused[a:a + step], bias, freq, 1.0, pos[a:a + step], seq[a:a + step], table, k, v, nh, nkv, d, layout)
             for a in range(0, M, step)]
        return torch.cat(q), k, v

    assert M * nkv * d >= 1 << 21 > 1000 * nkv * d  # one step takes the launch of its own, steps of 1,000 tokens do not
    for whole, parts in zip(run(M), run(1000)):
        assert torch.equal(whole, parts)
