"""The bfloat16 product of few rows where its rows of W are spread over all compute units, around the sizes at which the rule
changes, against 64 bits."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 3, 15, 576, 1040, 1041, 4096, 4097])
@pytest.mark.parametrize("K", [8, 1040, 2048, 4160])
def test_rows_spread_over_the_units(N, K):
    from pytorch_transformers_amd import ops

    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(64, K, generator=g).bfloat16().cuda()
    w = torch.randn(N, K, generator=g).bfloat16().cuda()
    want = x.double() @ w.double().T
    # 32-bit sums of products of bfloat16 numbers, which are exact: sqrt(K) roundings of partial sums of size sqrt(K)
    tol = 8 * 2.0 ** -24 * K + 1e-6
    whole = ops.gemm_skinny_bf16(x, w, out_f32=True)
    assert (whole.double() - want).abs().max().item() <= tol
    for m in (1, 8, 16, 17, 33, 48):
        assert torch.equal(ops.gemm_skinny_bf16(x[:m].contiguous(), w, out_f32=True), whole[:m])


@pytest.mark.parametrize("layout,nh,nkv,d", [("interleaved", 13, 13, 80), ("grouped", 4, 2, 6), ("tail", 7, 1, 64), ("grouped", 8, 2, 128), ("tail", 1, 1, 2)])
@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("rotation", ["none", "half", "interleaved part", "per sequence"])
def test_fused_rows_to_their_end(layout, nh, nkv, d, M, rotation):
    """The fused product on its own with the tail in its epilogue against the product and the kernel that splits, rotates and
    writes: the same bits (K no multiple of 2,048), nothing written elsewhere, nothing at all with write_cache off."""
    from pytorch_transformers_amd import ops

    if not ops.QKV_TAIL:
        pytest.skip("switched off by PTA_QKV_TAIL=0")
    K, N = 264, (nh + 2 * nkv) * d
    g = torch.Generator().manual_seed(M + d)
    r = lambda *s: torch.randn(*s, generator=g).cuda()
    x, w, bias = r(M, K).bfloat16(), (0.05 * r(N, K)).bfloat16(), r(N)
    part = d // 2 if rotation == "interleaved part" and d >= 4 else d
    part -= part % 2
    how = dict(rotary_dim=part, pairing="interleaved") if rotation == "interleaved part" else {}
    inv = None if rotation == "none" else 10000.0 ** (-torch.arange(part // 2, device="cuda").float() * 2 / part)
    if rotation == "per sequence":
        inv = (inv[None] * torch.arange(1, M + 1, device="cuda")[:, None]).contiguous()
    pos = torch.randint(0, 190, (M,), generator=g).int().cuda()
    seq, table = torch.arange(M).int().cuda(), torch.randperm(3 * M, generator=g).view(M, 3).int().cuda()
    assert ops.gemm_skinny_qkv_ok(x, w, d)
    new = lambda: (torch.full((3 * M, nkv, 64, d), 7.0).bfloat16().cuda(), torch.full((3 * M, nkv, d, 64), 7.0).bfloat16().cuda())
    k0, v0 = new()
    q0 = ops.qkv_rope_cache(ops.gemm_skinny_bf16(x, w), bias, inv, 0.9, pos, seq, table, k0, v0, nh, nkv, d, layout, **how)
    k1, v1 = new()
    q1 = ops.gemm_skinny_qkv(x, w, bias, inv, 0.9, pos, seq, table, k1, v1, nh, nkv, d, layout, True, **how)
    assert torch.equal(q0, q1) and torch.equal(k0, k1) and torch.equal(v0, v1)
    k2, v2 = new()
    ops.gemm_skinny_qkv(x, w, bias, inv, 0.9, pos, seq, table, k2, v2, nh, nkv, d, layout, False, **how)
    assert bool((k2 == 7.0).all()) and bool((v2 == 7.0).all())


# heads so short that a workgroup's rotation pairs (four up to N = 2,048, then eight) lie in three heads and more; of 12 in two
@pytest.mark.parametrize("layout,nh,nkv,d", [("grouped", 171, 171, 2), ("tail", 1026, 1, 2), ("grouped", 171, 171, 4), ("grouped", 256, 256, 4), ("tail", 340, 1, 6),
                                             ("grouped", 129, 129, 8), ("tail", 383, 1, 8), ("tail", 306, 1, 10), ("tail", 170, 1, 12)])
@pytest.mark.parametrize("rotation", ["none", "half", "interleaved part"])
def test_fused_rows_of_short_heads(layout, nh, nkv, d, rotation):
    test_fused_rows_to_their_end(layout, nh, nkv, d, 5, rotation)


LONG = (1 << 20) + 8  # elements of a row beyond what the launches through LDS address


# heads of one tile a workgroup, whose halves are eight rows, and of sixteen
@pytest.mark.parametrize("layout,nh,nkv,d", [("tail", 4, 1, 6), ("tail", 30, 1, 66)])
def test_fused_rows_of_very_long_rows(layout, nh, nkv, d):
    """The fused product taken to its end where rows of W go by registers: queries and cache pages within the product's rounding."""
    from pytorch_transformers_amd import ops

    if not ops.QKV_TAIL:
        pytest.skip("switched off by PTA_QKV_TAIL=0")
    M, N = 3, (nh + 2 * nkv) * d
    g = torch.Generator(device="cuda").manual_seed(d)
    x, w = torch.randn(M, LONG, generator=g, device="cuda").bfloat16(), torch.randn(N, LONG, generator=g, device="cuda").bfloat16()
    pos, seq, table = (torch.tensor(v, dtype=torch.int32, device="cuda") for v in ([5, 70, 130], [0, 1, 2], [[0, 1, 2], [3, 4, 5], [6, 7, 8]]))
    assert ops.gemm_skinny_qkv_ok(x, w, d)
    new = lambda: (torch.full((9, nkv, 64, d), 7.0).bfloat16().cuda(), torch.full((9, nkv, d, 64), 7.0).bfloat16().cuda())
    k0, v0 = new()
    q0 = ops.qkv_rope_cache(ops.gemm_skinny_bf16(x, w), None, None, 1.0, pos, seq, table, k0, v0, nh, nkv, d, layout)
    k1, v1 = new()
    q1 = ops.gemm_skinny_qkv(x, w, None, None, 1.0, pos, seq, table, k1, v1, nh, nkv, d, layout, True)
    for got, want in ((q1, q0), (k1, k0), (v1, v0)):  # sums in another order: a neighbour where they are rounded, the sums' roundings beside
        got, want = got.float(), want.float()
        assert ((got - want).abs() <= 2.0 ** -7 * want.abs() + 8 * 2.0 ** -24 * LONG).all()
    assert bool((k1 == 7.0).eq(k0 == 7.0).all()) and bool((v1 == 7.0).eq(v0 == 7.0).all())


def test_the_gate_of_very_long_rows():
    """As test_the_gate_in_the_epilogue, by registers."""
    from pytorch_transformers_amd import ops

    M, F = 2, 24
    g = torch.Generator(device="cuda").manual_seed(0)
    x, w = torch.randn(M, LONG, generator=g, device="cuda").bfloat16(), (0.002 * torch.randn(2 * F, LONG, generator=g, device="cuda")).bfloat16()
    assert ops.gemm_skinny_glu_ok(x, w)
    got = ops.gemm_skinny_glu(x, w, "silu", 1.7, 3.0).float()
    both = ops.gemm_skinny_bf16(x, w).float()
    gate, up = both[:, :F], both[:, F:]
    want = torch.nn.functional.silu(gate) * up
    # a neighbour of either half, and the sums' roundings at values of some 0.002 sqrt(K) = 2
    tol = 2.0 ** -7 * (1.3 * gate.abs() * (up.abs() + 1) + gate.abs() * up.abs() + want.abs()) + 1e-3
    assert bool(((got - want).abs() <= tol).all())


@pytest.mark.parametrize("M,N,K", [(1, 40, 72), (8, 8192, 2048), (16, 1048, 520)])
def test_squared_relu_in_the_epilogue(M, N, K):
    """Bias, squared ReLU and an addition in the launch itself: the bits of the product with its bias, taken to its end by hand."""
    from pytorch_transformers_amd import ops

    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), torch.randn(N, K, generator=g).bfloat16().cuda()
    bias, add = torch.randn(N, generator=g).cuda(), torch.randn(M, N, generator=g).bfloat16().cuda()
    z = ops.gemm_skinny_bf16(x, w, bias).float().clamp_min(0)
    assert torch.equal(ops.gemm_skinny_bf16(x, w, bias, "relu2"), (z * z).bfloat16())
    want = (z.double() * z.double() + add.double()).float()  # one rounding at the end, whether or not the two are one instruction
    got = ops.gemm_skinny_bf16(x, w, bias, "relu2", add)
    assert bool(((got.float() - want).abs() <= want.abs() * 2.0 ** -8 + z * z * 2.0 ** -23).all())


@pytest.mark.parametrize("kind", ["silu", "gelu_tanh", "clamped"])
@pytest.mark.parametrize("M,F,K", [(1, 1, 8), (16, 15, 72), (2, 5504, 2048), (9, 1040, 1040), (16, 4099, 264)])
def test_the_gate_in_the_epilogue(kind, M, F, K):
    """The gate of a feed-forward in the launch of its input product against the product and the gate's own launch.  Sums may
    be taken in another order (a half is then rounded to its neighbour), nothing else differs."""
    from pytorch_transformers_amd import ops

    g = torch.Generator().manual_seed(M + F)
    x, w = torch.randn(M, K, generator=g).bfloat16().cuda(), (0.05 * torch.randn(2 * F, K, generator=g)).bfloat16().cuda()
    assert ops.gemm_skinny_glu_ok(x, w)
    got = ops.gemm_skinny_glu(x, w, kind, 1.7, 3.0)
    both = ops.gemm_skinny_bf16(x, w)
    want = ops.glu(both[:, :F], both[:, F:], kind, 1.7, 3.0).float()
    gate, up = both[:, :F].float(), both[:, F:].float()
    # a neighbour of either half is 2^-7 of it away at most; the gates' slopes stay under 1.2 (1.3 at alpha 1.7)
    tol = 2.0 ** -7 * (1.3 * gate.abs() * (up.abs() + 1) + gate.abs() * up.abs() + want.abs()) + 1e-6
    assert bool(((got.float() - want).abs() <= tol).all())
    assert (got.float() != want).float().mean() <= 0.05


@pytest.mark.parametrize("F,K,fused", [(8, 64, False), (1024, 1024, False), (1032, 1024, True), (1536, 2048, True), (1536, 2056, False), (2048, 2056, False),
                                       (2056, 2056, True), (5504, 2048, True)])
@pytest.mark.parametrize("M", [1, 16])
def test_where_the_gate_rides_in_the_launch(monkeypatch, F, K, fused, M):
    """A feed-forward of 256 compute units' sizes: small matrices keep the product that spreads its rows over all of them."""
    from pytorch_transformers_amd import ops
    from pytorch_transformers_amd.parts import GatedFeedForward

    if ops.compute_units() != 256:
        pytest.skip("the lines are multiples of the compute units")
    g = torch.Generator().manual_seed(M + F)
    ff = GatedFeedForward("f", K, F)
    draw = {s.name: (0.05 * torch.randn(*s.shape, generator=g)).bfloat16().cuda() for s in ff.all_tensor_specs()}
    ff.load_all(draw)
    ff.after_load()
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    seen, call = [], ops._call
    monkeypatch.setattr(ops, "_call", lambda name, *a: (seen.append(name), call(name, *a))[1])
    got = ff.forward(x, None)
    assert seen[:-1] == (["pta_gemm_skinny_glu_bf16"] if fused else ["pta_gemm_skinny_bf16", "pta_glu"])
    both = ff.inp(x)
    want = ff.down(ops.glu(both[:, :F], both[:, F:])).float()
    assert (got.float() - want).norm() <= 2.0 ** -7 * want.norm()


@pytest.mark.parametrize("kind", ["silu", "gelu_tanh", "clamped"])
@pytest.mark.parametrize("F", [2052, 2057, 2064])
def test_one_arithmetic_of_the_gate_for_any_rows(kind, F):
    """A gate has the exponential of its own launch, which is another for rows that are no multiple of eight elements: sixteen
    rows of a feed-forward are formed as seventeen are."""
    from pytorch_transformers_amd import ops

    g = torch.Generator().manual_seed(F)
    x, w = torch.randn(17, 64, generator=g).bfloat16().cuda(), torch.randn(2 * F, 64, generator=g).bfloat16().cuda()
    assert ops.gemm_skinny_glu_pays(x[:16], w) == (F % 8 == 0)
    if F % 8 == 0:  # the same exponential on both sides: what differs is the product's sums
        both = ops.gemm_skinny_bf16(x[:16], w)
        got, want = ops.gemm_skinny_glu(x[:16], w, kind, 1.7, 3.0), ops.glu(both[:, :F], both[:, F:], kind, 1.7, 3.0)
        assert (got != want).float().mean() <= 0.01


@pytest.mark.parametrize("act", ["relu2", "silu", "gelu_new"])
@pytest.mark.parametrize("N", [64, 8192])
def test_activations_of_32_bit_results_are_refused(act, N):
    """Results in 32-bit are the output head's: they take no activation but the exact GELU."""
    from pytorch_transformers_amd import ops

    x, w = torch.ones(2, 64).bfloat16().cuda(), torch.ones(N, 64).bfloat16().cuda()
    with pytest.raises(ops.KernelError, match="needs a bfloat16 result"):
        ops.gemm_skinny_bf16(x, w, act=act, out_f32=True)
    assert torch.equal(ops.gemm_skinny_bf16(x, w, act=act, out_f32=False), ops.epilogue_(ops.gemm_skinny_bf16(x, w), None, act))
