"""The 32-bit kernels alone, against 64-bit references: every way a product runs (few rows, tiles, shared segments),
at the edges of their tiles, and the same bits for a row whichever of them it runs in."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from pytorch_transformers_amd import ops

    ops.load_library()
    return ops


def _rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).cuda()


@pytest.mark.parametrize("N,K", [(1, 1), (40, 15), (129, 16), (260, 100), (64, 1040), (4544, 576), (8200, 300), (96, 2050)])
def test_products(N, K):
    """Rows 1 .. 700 (few rows with one, two and four tiles; 64 and 128 tiles; shared segments), K with and without a last
    block and rows that are no multiple of sixteen bytes."""
    ops = _ops()
    M = 700
    a, w, bias, a1, a2 = _rand(M, K), _rand(N, K, seed=1), _rand(N, seed=2), _rand(M, N, seed=3), _rand(M, N, seed=4)
    prod = a.double() @ w.double().T
    # |error| <= K eps sum |a w| in the worst case; the sums are of random signs, so sqrt(K) eps times the root of the sum of squares
    scale = ((a.double() ** 2) @ (w.double() ** 2).T).sqrt().max().item()
    tol = 8 * 2.0 ** -24 * math.sqrt(K) * scale + 1e-30
    plain = ops.gemm_f32(a, w)
    assert (plain.double() - prod).abs().max().item() <= tol
    v = prod + bias.double()
    want = 0.5 * v * (1 + torch.erf(v / math.sqrt(2.0))) + a1.double() + a2.double()
    full = ops.gemm_f32(a, w, bias, "gelu", a1, a2)
    assert (full.double() - want).abs().max().item() <= 2 * tol + 2e-6 * want.abs().max().item()
    for m in (1, 2, 16, 17, 33, 64, 65, 128, 300):
        assert torch.equal(ops.gemm_f32(a[:m].contiguous(), w), plain[:m]), f"{m} rows alone and in a batch"
        assert torch.equal(ops.gemm_f32(a[:m].contiguous(), w, bias, "gelu", a1[:m].contiguous(), a2[:m].contiguous()), full[:m])
