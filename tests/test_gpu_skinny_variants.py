"""Every variant of the few-row product at matrices that its workgroups share evenly and unevenly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("N", [4096, 8192, 16384, 4095, 16448])
def test_variants_give_the_product(N, variant):
    """64 rows of W for each workgroup (variants 3 and 4 at N = 4,096 and its multiples) down to a few, with rows of x of each class."""
    from pytorch_transformers_amd import ops

    K = 72
    g = torch.Generator(device="cuda").manual_seed(N + variant)
    w = torch.randn((N, K), generator=g, device="cuda").bfloat16()
    for M in (1, 16, 17, 33, 64):
        x = torch.randn((M, K), generator=g, device="cuda").bfloat16()
        want = x.float() @ w.float().t()
        got = ops.gemm_skinny_bf16(x, w, out_f32=True, variant=variant)
        # sums of K products of bfloat16 values in 32 bits, in any order: K rounding steps of the absolute sum at most
        bound = K * 2.0 ** -24 * 2 * (x.float().abs() @ w.float().abs().t())
        assert bool(((got - want).abs() <= bound).all()), f"{M} rows: off by {float((got - want).abs().max())}"
