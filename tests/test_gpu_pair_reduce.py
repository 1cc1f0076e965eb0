"""The reduction of a pair whose first product is a query_key_value projection: the second product's elements four a thread, and one where rows are no
multiple of four."""
import pytest
import torch

from pytorch_transformers_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N2,K2", [(17, 4, 64), (17, 530, 64), (33, 1032, 2112), (48, 95, 1544), (64, 4096, 512)])
@pytest.mark.parametrize("bias,act", [(False, None), (True, "gelu")])
def test_the_second_product_is_the_plain_pair_s(M, N2, K2, bias, act):
    """The same operations on the same sums: the same bits."""
    g = torch.Generator().manual_seed(M + N2)
    nh, nkv, d, K1 = 4, 1, 32, 512
    draw = lambda *shape: (torch.randn(shape, generator=g) * 0.2).bfloat16().cuda()
    x1, w1, x2, w2 = draw(M, K1), draw((nh + 2 * nkv) * d, K1), draw(M, K2), draw(N2, K2)
    b2 = torch.randn(N2, generator=g).cuda() if bias else None
    pools = [torch.zeros((M + 1, nkv, 64, d), dtype=torch.bfloat16, device="cuda"), torch.zeros((M + 1, nkv, d, 64), dtype=torch.bfloat16, device="cuda")]
    pos, seq = torch.arange(M, dtype=torch.int32).cuda() % 64, torch.arange(M, dtype=torch.int32).cuda()
    table = torch.arange(1, M + 1, dtype=torch.int32).view(M, 1).cuda()
    inv = (10000.0 ** (-torch.arange(0, d, 2) / d)).cuda()
    q, y2 = ops.gemm_splitk_pair_qkv(x1, w1, None, inv, 1.0, pos, seq, table, *pools, nh, nkv, d, "grouped", True, x2, w2, b2, act)
    y1, want = ops.gemm_splitk_pair_bf16(x1, w1, x2, w2, None, None, b2, act)
    assert torch.equal(y2, want)
    assert torch.isfinite(q).all() and y1.shape == (M, (nh + 2 * nkv) * d)
