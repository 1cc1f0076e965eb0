"""The few-row product whose tiles are eight rows of W at two places of K: the sizes around which its rules change, against 64
bits, and the same bits for any number of rows of x."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [5, 1023, 2047, 2048, 2049])
@pytest.mark.parametrize("K", [8, 56, 64, 72, 120, 128, 136, 264, 1040, 8192])
def test_eight_rows_at_two_places_of_k(N, K):
    from pytorch_transformers_amd import ops

    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(16, K, generator=g).bfloat16().cuda()
    w = torch.randn(N, K, generator=g).bfloat16().cuda()
    bias, add = torch.randn(N, generator=g).cuda(), torch.randn(16, N, generator=g).bfloat16().cuda()
    want = x.double() @ w.double().T
    whole = ops.gemm_skinny_bf16(x, w, out_f32=True)
    tol = 8 * 2.0 ** -24 * K + 1e-6  # 32-bit sums of exact products: sqrt(K) roundings of partial sums of size sqrt(K)
    assert (whole.double() - want).abs().max().item() <= tol
    for m in (1, 7, 8, 9, 15):
        assert torch.equal(ops.gemm_skinny_bf16(x[:m].contiguous(), w, out_f32=True), whole[:m])
    got = ops.gemm_skinny_bf16(x[:7].contiguous(), w, bias, None, add[:7].contiguous())
    by_hand = ((whole[:7].bfloat16().float() + bias).bfloat16().float() + add[:7].float()).bfloat16()
    assert torch.equal(got, by_hand)
