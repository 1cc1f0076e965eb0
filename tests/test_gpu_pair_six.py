"""Pairs of products on workgroups of six waves (96 rows of W): the edges of their tiles, ranges and rows of x."""
import pytest
import torch

from pytorch_transformers_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [33, 47, 48, 49, 64])
@pytest.mark.parametrize("N1,K1,N2,K2,p1,p2", [(4096, 64, 96, 200, 1, 1), (4001, 1032, 95, 1544, 2, 3), (2049, 2048, 2111, 4096, 1, 4), (97, 72, 4008, 72, 1, 1)])
def test_six_waves_are_four(N1, K1, N2, K2, p1, p2, rows):
    """The height of a tile changes no sum (the bits of workgroups of four waves with the same ranges) but where rows are a multiple of 4 KB long: there
    each tile walks K from a place of its own."""
    g = torch.Generator().manual_seed(N1 + rows)
    draw = lambda *shape: torch.randn(shape, generator=g).bfloat16().cuda()
    x1, w1, x2, w2 = draw(rows, K1), draw(N1, K1), draw(rows, K2), draw(N2, K2)
    lib, out = ops.load_library(), []
    try:
        for kind in (1, 2, 4):
            assert lib.pta_gemm_splitk_pair_fix_middle(N1, K1, N2, K2, p1, p2, kind) == 0
            assert ops.gemm_splitk_pair_way(N1, K1, N2, K2, rows) == (p1, p2, kind)
            out.append(ops.gemm_splitk_pair_partial(x1, w1, x2, w2))
    finally:
        lib.pta_gemm_splitk_pair_fix(N1, K1, N2, K2, 0, 0, 1)
    if K1 % 2048 and K2 % 2048:
        for kind in out[1:]:
            assert torch.equal(kind[0], out[0][0]) and torch.equal(kind[1], out[0][1])
    for part, x, w in zip(out[2], (x1, x2), (w1, w2)):
        want = x.double() @ w.double().t()
        size = x.double().abs() @ w.double().abs().t()
        assert ((part.double().sum(0) - want).abs() <= 2.0 ** -24 * x.shape[1] * size).all()  # K additions in 32-bit


def test_beyond_64_rows_they_are_not_taken():
    lib, shape = ops.load_library(), (4096, 512, 512, 512)
    try:
        assert lib.pta_gemm_splitk_pair_fix(*shape, 1, 1, 4) == 0
        assert [ops.gemm_splitk_pair_way(*shape, rows)[2] for rows in (8, 32, 33, 64, 150)] == [1, 1, 4, 4, 1]
        assert lib.pta_gemm_splitk_pair_fix_middle(*shape, 1, 1, 3) == 1 and lib.pta_gemm_splitk_pair_fix_middle(*shape, 1, 1, 5) == 1
    finally:
        lib.pta_gemm_splitk_pair_fix(*shape, 0, 0, 1)
