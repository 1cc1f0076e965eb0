"""The norm that goes on to the weighted sum of streams: counts of planes around those that are asked for ahead, one and two pieces a thread."""
import pytest
import torch

from pytorch_transformers_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,gated,groups", [(3, 512, False, 1), (5, 4096, True, 2), (2, 4100, False, 1), (3, 8192, True, 1)])
@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 6, 8, 9, 12])
def test_norm_and_sum_are_the_two_launches(rows, width, gated, groups, count, dtype):
    """Both form the sum in the order of the planes; they may contract its products otherwise."""
    g = torch.Generator().manual_seed(width + count)
    x, res, w = torch.randn(rows, width, generator=g).to(dtype).cuda(), torch.randn(rows, width, generator=g).cuda(), torch.randn(width, generator=g).cuda()
    gate = torch.randn(rows, width, generator=g).to(dtype).cuda() if gated else None
    planes, coef = torch.randn(count + 1, rows, width, generator=g).cuda(), torch.randn(count, generator=g).cuda()
    how = dict(residual=res, mult=0.5, gate=gate, groups=groups)
    two = planes.clone()
    ops.rmsnorm(x, w, 1e-5, dtype, want_narrow=False, out_wide=two[count - 1], **how)
    narrow, wide = ops.depth_mix(two, coef, count, dtype)
    got_narrow, got_wide = ops.rmsnorm(x, w, 1e-5, dtype, out_wide=planes[count - 1], mix=(planes, coef, count), **how)
    # the norm's own plane by the same operations, contracted otherwise at most; none of the others
    torch.testing.assert_close(planes[count - 1], two[count - 1], rtol=1e-6, atol=1e-6 * two[count - 1].abs().max().item())
    keep = [j for j in range(count + 1) if j != count - 1]
    assert torch.equal(planes[keep], two[keep])
    # count products and sums in 32-bit on each side
    size = (coef[:, None, None].abs() * two[:count].abs()).sum(0)
    bound = 2 * count * 2.0 ** -24 * size + 2e-6 * coef[-1].abs() * two[count - 1].abs().max()
    assert ((got_wide - wide).abs() <= bound).all()
    assert ((got_narrow.float() - narrow.float()).abs() <= bound + (0 if dtype == torch.float32 else 2.0 ** -8) * wide.abs()).all()
