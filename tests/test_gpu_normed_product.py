"""The product of few rows with the LayerNorm in front of it in one launch, against 64 bits and against the launches it stands
for, at the edges of its sizes."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _on():
    from pytorch_transformers_amd import ops

    if not ops.GEMM_NORMED:
        pytest.skip("switched off by PTA_GEMM_NORMED=0")


def _draw(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g).cuda()
    x = (r(M, K) * 3 + 1).bfloat16()
    return x, (0.05 * r(N, K)).bfloat16(), 1 + 0.2 * r(K), 0.2 * r(K), r(N)


@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(1, 8), (17, 64), (300, 504), (4160, 512), (1040, 520), (4160, 1040), (2304, 768), (8192, 2048), (33, 2040)])
@pytest.mark.parametrize("act", [None, "gelu", "silu"])
def test_norm_and_product(M, N, K, act):
    from pytorch_transformers_amd import ops

    x, w, gain, shift, bias = _draw(M, N, K, M + N + K)
    assert ops.gemm_normed_ok(x, w)
    got = ops.gemm_normed(x, gain, shift, 1e-5, w, bias, act).double()
    rows = torch.nn.functional.layer_norm(x.double(), (K,), gain.double(), shift.double(), 1e-5).bfloat16().double()
    z = rows @ w.double().T
    z = (z.bfloat16().double() + bias.double()).bfloat16().double()
    want = z if act is None else getattr(torch.nn.functional, act)(z)
    # normed rows may be rounded to the neighbour where 32-bit statistics are a little off (2^-8 of an element, in few places);
    # the product and the sum with the bias are rounded to 2^-8 of themselves each
    size = (rows.abs() @ w.double().abs().T).max()
    tol = 2.0 ** -7 * (z.abs() + bias.double().abs()) + 2.0 ** -8 * size / K ** 0.5 + 2.0 ** -8 * want.abs() + 1e-6
    assert bool(((got - want).abs() <= 1.2 * tol).all())
    assert (got - want).norm() <= 2.0 ** -8 * want.norm() + 1e-6
    plain = ops.gemm_skinny_bf16(ops.layernorm(x, gain, shift, 1e-5), w, bias, act).double()
    assert (plain - got).norm() <= 2.0 ** -8 * want.norm() + 1e-6


@pytest.mark.parametrize("layout,nh,nkv,d", [("interleaved", 13, 13, 80), ("grouped", 4, 2, 6), ("tail", 7, 1, 64), ("tail", 1, 1, 2)])
@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("rotated", [False, True])
def test_norm_and_fused_rows_to_their_end(layout, nh, nkv, d, M, rotated):
    """Queries and cache of the launch with the norm in it against the norm and the launch without: what differs comes from a
    normed element rounded to its neighbour."""
    from pytorch_transformers_amd import ops

    K, N = 1040, (nh + 2 * nkv) * d
    x, w, gain, shift, bias = _draw(M, N, K, M + d)
    g = torch.Generator().manual_seed(d)
    inv = 10000.0 ** (-torch.arange(d // 2, device="cuda").float() * 2 / d) if rotated else None
    pos = torch.randint(0, 190, (M,), generator=g).int().cuda()
    seq, table = torch.arange(M).int().cuda(), torch.randperm(3 * M, generator=g).view(M, 3).int().cuda()
    new = lambda: (torch.full((3 * M, nkv, 64, d), float("nan")).bfloat16().cuda(), torch.full((3 * M, nkv, d, 64), float("nan")).bfloat16().cuda())
    k0, v0 = new()
    q0 = ops.gemm_skinny_qkv(ops.layernorm(x, gain, shift, 1e-5), w, bias, inv, 0.9, pos, seq, table, k0, v0, nh, nkv, d, layout, True)
    k1, v1 = new()
    q1 = ops.gemm_normed_qkv(x, gain, shift, 1e-5, w, bias, inv, 0.9, pos, seq, table, k1, v1, nh, nkv, d, layout, True)
    page, at = table[torch.arange(M, device="cuda"), (pos // 64).long()].long(), (pos % 64).long()
    rows = lambda k, v: (k[page, :, at], v[page, :, :, at])  # what each token wrote
    for a, b in zip((q0,) + rows(k0, v0), (q1,) + rows(k1, v1)):
        a, b = a.float(), b.float()
        # sums of ~1,000 terms of which a few normed ones are a neighbour (2^-8 of themselves), the results a neighbour in places
        assert bool(torch.isfinite(a).all()) and (a - b).norm() <= 2.0 ** -8 * a.norm()
        assert (a - b).abs().max() <= 2.0 ** -6 * a.abs().max()
    for pool in (k1, v1):  # and nothing else
        assert int((~pool.isnan()).sum()) == M * nkv * d
    k2, v2 = new()
    ops.gemm_normed_qkv(x, gain, shift, 1e-5, w, bias, inv, 0.9, pos, seq, table, k2, v2, nh, nkv, d, layout, False)
    assert bool(k2.isnan().all()) and bool(v2.isnan().all())


def test_sizes_it_leaves_to_others():
    from pytorch_transformers_amd import ops

    ok = lambda M, N, K: ops.gemm_normed_ok(torch.empty(M, K, dtype=torch.bfloat16, device="cuda"), torch.empty(N, K, dtype=torch.bfloat16, device="cuda"))
    assert ok(8, 8192, 2048) and ok(16, 4096, 2048) and ok(16, 8192, 2048) and not ok(17, 64, 64) and not ok(1, 64, 2056) and not ok(1, 64, 12) and not ok(1, 8193, 64)


@pytest.mark.parametrize("N,K", [(64, 64), (4096, 2048), (4352, 1040), (4368, 1536), (8192, 520), (8192, 2048)])
def test_a_row_has_the_same_bits_in_any_batch(N, K):
    """Sizes of W alone choose the launch, its waves and so the order of summation: of sixteen rows each is what it is alone."""
    from pytorch_transformers_amd import ops

    x, w, gain, shift, bias = _draw(16, N, K, N + K)
    assert all(ops.gemm_normed_ok(x[:m], w) for m in (1, 8, 9, 16))
    whole = ops.gemm_normed(x, gain, shift, 1e-5, w, bias, "gelu")
    for rows in (x[:1], x[:8], x[:9], x[:13]):
        assert torch.equal(ops.gemm_normed(rows, gain, shift, 1e-5, w, bias, "gelu"), whole[:len(rows)])
    assert torch.equal(ops.gemm_normed(x[9:10].contiguous(), gain, shift, 1e-5, w, bias, "gelu"), whole[9:10])


@pytest.mark.parametrize("which", ["mixer", "feed-forward", "no product"])
def test_parts_that_read_their_input_get_the_normed_rows(which):
    """A mixer or feed-forward with a ``forward`` of its own may read its input beside the product that it is handed: what it is
    given is the norm's result then; the library's own parts, which read nothing else, have the norm inside the product's launch."""
    import test_gpu_parts as TP
    from pytorch_transformers_amd import ops
    from pytorch_transformers_amd.cache import PagedCache
    from pytorch_transformers_amd.engine.spec import CACHE_FULL, CacheGroupSpec, LayerCall
    from pytorch_transformers_amd.parts import AttentionMixer, DenseFeedForward, LayerNorm, NoPositions, SequentialBlock
    from pytorch_transformers_amd.parts.base import as_tensor

    H, nh, d, seen = 64, 4, 16, []

    class OwnMixer(AttentionMixer):
        def forward(self, x, *a, **k):
            seen.append(x)
            return super().forward(x, *a, **k)

    class OwnFeedForward(DenseFeedForward):
        def forward(self, x, *a, **k):
            seen.append(x)
            return super().forward(x, *a, **k)

    class NoProduct(DenseFeedForward):
        def input_projection(self):
            return None, {}

    def block(mixer, ffn):
        b = SequentialBlock(mixer("a", H, nh, nh, d, "interleaved", True, NoPositions()), ffn("f", H, 128, bias=True), LayerNorm("n1", H, 1e-5),
                            LayerNorm("n2", H, 1e-5))
        TP._fill(b, torch.bfloat16, 3)
        return b

    x = torch.randn(3, H, generator=torch.Generator().manual_seed(0)).bfloat16().cuda()

    def run(b):
        cache = PagedCache([CacheGroupSpec("kv", CACHE_FULL, 1, nh, d)], 256, torch.bfloat16, "cuda:0")
        ctx, _ = TP._ctx(cache, [cache.alloc()], [3], torch.bfloat16)
        return as_tensor(b.forward(x, ctx, LayerCall(0, "kv", 0))).float()

    want = run(block(AttentionMixer, DenseFeedForward))
    b = block(OwnMixer if which == "mixer" else AttentionMixer, {"feed-forward": OwnFeedForward, "no product": NoProduct}.get(which, DenseFeedForward))
    got = run(b)
    assert (got - want).norm() <= 2.0 ** -7 * want.norm()
    if which == "mixer":
        assert torch.equal(seen[0], b.norm_in.forward(x))
    elif which == "feed-forward":
        a = seen[0].float()  # rows of a norm: the gain and shift taken off, mean 0 and mean square 1
        z = (a - b.norm_post.bias) / b.norm_post.weight
        assert z.mean(1).abs().max() <= 0.02 and (z.pow(2).mean(1) - 1).abs().max() <= 0.05
