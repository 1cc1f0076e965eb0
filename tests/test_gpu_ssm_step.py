"""A decode step of the state-space mixer in one launch against the launches that it takes the place of."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _both(seqs, heads, groups, N, K, dtype, apart=8):
    """A step's rows, table and slots by the launches one after the other and by the one: (rows, moved table) of each, the table before and the slots."""
    from pytorch_transformers_amd import ops

    g = torch.Generator(device="cuda").manual_seed(heads * N + K)
    draw = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    inner = heads * 64
    C, cut = inner + 2 * groups * N, heads * N * 64
    table = draw(seqs + 3, cut + (K - 1) * C + 8 - ((K - 1) * C) % 4)[:, :cut + (K - 1) * C]
    assert ops.ssm_step_ok(table, heads, 64, N, groups, K, groups)
    proj = draw(seqs, inner + C + heads + apart).to(dtype)[:, :inner + C + heads]
    w, b, dt_b, a_log, d, nw = draw(C, K), draw(C), draw(heads), draw(heads), draw(heads), draw(inner)
    slots = torch.randperm(seqs + 3, generator=torch.Generator().manual_seed(1))[:seqs].to(torch.int32).cuda()
    cu = torch.arange(seqs + 1, dtype=torch.int32, device="cuda")
    one, two = table.clone(), torch.empty_strided(table.shape, table.stride(), device="cuda")
    two.copy_(table)
    xbc = ops.conv_silu(proj[:, inner:inner + C], w, b, one[:, cut:], cu, cu[:-1].contiguous(), slots)
    y = ops.ssm_scan(xbc, proj[:, inner + C:], dt_b, a_log, d, one[:, :cut], cu, slots, heads, 64, N, groups)
    want = ops.rmsnorm(y, nw, 1e-6, dtype, offset=1.0, groups=groups, gate=proj[:, :inner])[0]
    got = ops.ssm_step(proj, w, b, dt_b, a_log, d, two, nw, 1.0, 1e-6, cu, slots, heads, 64, N, groups)
    return (want, one), (got, two), table, slots


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seqs,heads,groups,N,K", [(8, 64, 8, 128, 4), (1, 8, 8, 64, 2), (3, 5, 5, 128, 3), (5, 6, 2, 64, 4), (2, 14, 2, 128, 4)])
def test_a_step_is_the_launches_one_after_the_other(seqs, heads, groups, N, K, dtype):
    """Groups of one head (whose threads form several channels each) up to eight, both heights of the state, all numbers of taps; rows of the table in
    no order and apart, rows of the product apart."""
    (want, one), (got, two), table, slots = _both(seqs, heads, groups, N, K, dtype)
    cut = heads * N * 64
    assert torch.equal(one[:, cut:], two[:, cut:])  # the tail is moved, not formed
    # sums of N terms in 32 bits: N rounding steps at most (the bits, where heads of a group are a power of two: below)
    torch.testing.assert_close(two[:, :cut], one[:, :cut], rtol=4e-6, atol=4e-6)
    tol = N * 2.0 ** -24 * 8 if dtype == torch.float32 else 2.0 ** -8
    torch.testing.assert_close(got.float(), want.float(), rtol=tol, atol=tol * want.float().abs().max().item())
    untouched = [i for i in range(seqs + 3) if i not in slots.tolist()]
    assert torch.equal(two[untouched], table[untouched])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seqs,heads,groups,N,K,apart", [(8, 64, 8, 128, 4, 8), (2, 16, 2, 64, 4, 8), (2, 16, 2, 64, 4, 7), (3, 5, 5, 128, 3, 8), (5, 6, 2, 64, 4, 8),
                                                         (1, 8, 2, 64, 2, 8), (2, 14, 2, 128, 4, 8)])
def test_a_step_leaves_the_bits_of_the_launches(seqs, heads, groups, N, K, apart, dtype):
    """A sequence that is walked in steps of one token by either way goes on from the same state: every order and contraction is the launches' own.  Groups
    of one to eight heads; eight with rows of the product that the norm reads four elements at a time, and (apart 7) with rows that it does not."""
    (want, one), (got, two), _, _ = _both(seqs, heads, groups, N, K, dtype, apart)
    assert torch.equal(one, two)
    assert torch.equal(want, got)


def test_sizes_that_keep_the_launches_apart():
    from pytorch_transformers_amd import ops

    table = torch.zeros((2, 1 << 20), device="cuda")
    assert ops.ssm_step_ok(table, 64, 64, 128, 8, 4, 8)
    for sizes in ((64, 64, 128, 8, 4, 1), (64, 32, 128, 8, 4, 8), (64, 64, 96, 8, 4, 8), (64, 64, 128, 4, 4, 4), (64, 64, 128, 8, 5, 8), (64, 64, 128, 8, 1, 8)):
        assert not ops.ssm_step_ok(table, *sizes)
    assert not ops.ssm_step_ok(table[:, 1:], 64, 64, 128, 8, 4, 8)
    assert not ops.ssm_step_ok(table[:, :99].contiguous(), 64, 64, 128, 8, 4, 8)
