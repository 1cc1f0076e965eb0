"""A decode step of the state-space mixer in one launch against the launches that it takes the place of."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seqs,heads,groups,N,K", [(8, 64, 8, 128, 4), (1, 8, 8, 64, 2), (3, 5, 5, 128, 3), (5, 6, 2, 64, 4), (2, 14, 2, 128, 4)])
def test_a_step_is_the_launches_one_after_the_other(seqs, heads, groups, N, K, dtype):
    """Groups of one head (whose threads form several channels each) up to eight, both heights of the state, all numbers of taps; rows of the table in
    no order and apart, rows of the product apart."""
    from pytorch_transformers_amd import ops

    g = torch.Generator(device="cuda").manual_seed(heads * N + K)
    draw = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    inner = heads * 64
    C, cut = inner + 2 * groups * N, heads * N * 64
    table = draw(seqs + 3, cut + (K - 1) * C + 8 - ((K - 1) * C) % 4)[:, :cut + (K - 1) * C]
    assert ops.ssm_step_ok(table, heads, 64, N, groups, K, groups)
    proj = draw(seqs, inner + C + heads + 8).to(dtype)[:, :inner + C + heads]
    w, b, dt_b, a_log, d, nw = draw(C, K), draw(C), draw(heads), draw(heads), draw(heads), draw(inner)
    slots = torch.randperm(seqs + 3, generator=torch.Generator().manual_seed(1))[:seqs].to(torch.int32).cuda()
    cu = torch.arange(seqs + 1, dtype=torch.int32, device="cuda")
    one, two = table.clone(), torch.empty_strided(table.shape, table.stride(), device="cuda")
    two.copy_(table)
    xbc = ops.conv_silu(proj[:, inner:inner + C], w, b, one[:, cut:], cu, cu[:-1].contiguous(), slots)
    y = ops.ssm_scan(xbc, proj[:, inner + C:], dt_b, a_log, d, one[:, :cut], cu, slots, heads, 64, N, groups)
    want = ops.rmsnorm(y, nw, 1e-6, dtype, offset=1.0, groups=groups, gate=proj[:, :inner])[0]
    got = ops.ssm_step(proj, w, b, dt_b, a_log, d, two, nw, 1.0, 1e-6, cu, slots, heads, 64, N, groups)
    assert torch.equal(one[:, cut:], two[:, cut:])  # the tail is moved, not formed
    # the same sums of N terms in 32 bits, which may be contracted otherwise: N rounding steps at most
    torch.testing.assert_close(two[:, :cut], one[:, :cut], rtol=4e-6, atol=4e-6)
    tol = N * 2.0 ** -24 * 8 if dtype == torch.float32 else 2.0 ** -8
    torch.testing.assert_close(got.float(), want.float(), rtol=tol, atol=tol * want.float().abs().max().item())
    untouched = [i for i in range(seqs + 3) if i not in slots.tolist()]
    assert torch.equal(two[untouched], table[untouched])


def test_sizes_that_keep_the_launches_apart():
    from pytorch_transformers_amd import ops

    table = torch.zeros((2, 1 << 20), device="cuda")
    assert ops.ssm_step_ok(table, 64, 64, 128, 8, 4, 8)
    for sizes in ((64, 64, 128, 8, 4, 1), (64, 32, 128, 8, 4, 8), (64, 64, 96, 8, 4, 8), (64, 64, 128, 4, 4, 4), (64, 64, 128, 8, 5, 8), (64, 64, 128, 8, 1, 8)):
        assert not ops.ssm_step_ok(table, *sizes)
    assert not ops.ssm_step_ok(table[:, 1:], 64, 64, 128, 8, 4, 8)
    assert not ops.ssm_step_ok(table[:, :99].contiguous(), 64, 64, 128, 8, 4, 8)
