"""Which kernel a product of a decode batch goes to: a captured step, padded to a multiple of eight rows, as the same step run directly
(no GPU)."""
import pytest


@pytest.mark.parametrize("N", [1024, 4096, 4104, 5000, 6000, 7280, 7288, 8000, 8064, 8192])
@pytest.mark.parametrize("K", [64, 256, 1024, 2560])
def test_small_products_long_in_n_of_padded_rows(N, K):
    from pytorch_transformers_amd import ops

    for M in range(17, 129):
        assert ops._splitk_small(M, N, K) == ops._splitk_small((M + 7) // 8 * 8, N, K), M
