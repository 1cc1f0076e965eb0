"""The product of many rows (``ops.gemm_tile_bf16``) against 64-bit products: edges of tiles, ends of K, every tile height, cut
and whole tiles, rows that lie apart, and what its epilogue adds."""
import pytest
import torch

from pytorch_transformers_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _draw(M, N, K, seed, ldx=None):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    x = torch.randn((M, ldx or K), generator=g, device=DEV).to(torch.bfloat16)[:, :K]
    return x, torch.randn((N, K), generator=g, device=DEV).to(torch.bfloat16)


def _check(got, x, w, K):
    """One rounding to bfloat16 (half of 2^-7 of the value below it) of a sum whose 32-bit additions are off by at most K 2^-24 of the
    sum of its terms' sizes each."""
    xd, wd = x.double(), w.double()
    want = xd @ wd.t()
    room = want.abs() * 2.0 ** -8 + (xd.abs() @ wd.abs().t()) * (K * 2.0 ** -24) * 1.01
    assert bool(((got.double() - want).abs() <= room).all()), float(((got.double() - want).abs() / room).max())


@pytest.mark.parametrize("fq", range(2, 9))
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (129, 264, 72), (300, 520, 1040), (513, 1000, 200)])
def test_tiles(M, N, K, fq):
    x, w = _draw(M, N, K, M + fq)
    tiles = -(-M // (32 * fq)) * -(-N // 256)
    blocks = -(-K // 64)
    plans = {(tiles, 1), (tiles // 2, min(2, blocks)), (0, min(3, blocks)), (0, blocks)}
    for whole, split in sorted(plans):
        _check(ops.gemm_tile_bf16(x, w, plan=(fq, whole, split)), x, w, K)


@pytest.mark.parametrize("M,N,K", [(129, 4672, 4544), (672, 4544, 18176), (895, 1040, 4160), (2048, 2048, 64), (1500, 18176, 128)])
def test_chosen_plan(M, N, K):
    x, w = _draw(M, N, K, N)
    _check(ops.gemm_tile_bf16(x, w), x, w, K)


def test_rows_apart():
    x, w = _draw(333, 640, 328, 5, ldx=800)
    assert not x.is_contiguous()
    for plan in (None, (4, 0, 3)):
        _check(ops.gemm_tile_bf16(x, w, plan=plan), x, w, 328)


@pytest.mark.parametrize("plan", [(3, 8, 1), (3, 4, 2), (8, 0, 4)])
@pytest.mark.parametrize("act", [None, "gelu", "relu2"])
def test_epilogue_is_the_one_of_a_pass_of_its_own(act, plan):
    """Bias, activation and additions on the rounded product: the same bits as ``epilogue_`` on the product alone."""
    M, N, K = 190, 1000, 320
    x, w = _draw(M, N, K, 9)
    bias = torch.randn(N, device=DEV) * 5
    add1, add2 = (torch.randn((M, N), device=DEV).to(torch.bfloat16) for _ in range(2))
    plan = (plan[0], min(plan[1], -(-M // (32 * plan[0])) * 4), plan[2])
    for b, a1, a2 in ((None, None, None), (bias, None, None), (bias, add1, None), (None, add1, add2), (bias, add1, add2)):
        want = ops.gemm_tile_bf16(x, w, plan=plan)
        if act or b is not None or a1 is not None:
            ops.epilogue_(want, b, act, a1, a2)
        got = ops.gemm_tile_bf16(x, w, b, act, a1, a2, plan=plan)
        assert torch.equal(got, want)


def test_infinite_rows_stay_their_own():
    """A row past the end of K or of a tile adds nothing: values that are not finite change no other row or column."""
    M, N, K = 130, 264, 72
    x, w = _draw(M, N, K, 3)
    clean = ops.gemm_tile_bf16(x, w, plan=(2, 0, 2))
    x2, w2 = x.clone(), w.clone()
    x2[7, 70] = float("inf")
    w2[263, 1] = float("nan")
    got = ops.gemm_tile_bf16(x2, w2, plan=(2, 0, 2))
    keep_r = torch.arange(M, device=DEV) != 7
    assert torch.equal(got[keep_r][:, :263], clean[keep_r][:, :263])
    assert not bool(torch.isfinite(got[7]).any()) and bool(torch.isnan(got[:, 263]).all())


@pytest.mark.parametrize("what", ["N", "K", "plan", "type"])
def test_refused(what):
    x, w = _draw(130, 264, 72, 1)
    with pytest.raises(ops.KernelError):
        if what == "N":
            ops.gemm_tile_bf16(x, w[:260], plan=(2, 0, 1))
        elif what == "K":
            ops.gemm_tile_bf16(x[:, :68], w[:, :68].contiguous(), plan=(2, 0, 1))
        elif what == "plan":
            ops.gemm_tile_bf16(x, w, plan=(9, 0, 1))
        else:
            ops.gemm_tile_bf16(x.float(), w)


def test_additions_at_any_address():
    """The kernel's epilogue adds sixteen bytes at a time; additions that lie elsewhere are added behind it, to the same bits."""
    M, N, K = 300, 264, 72
    x, w = _draw(M, N, K, 5)
    bias = torch.randn(N, generator=torch.Generator().manual_seed(6)).to(DEV)
    wide = torch.randn(2 * M * N + 1, generator=torch.Generator().manual_seed(7)).bfloat16().to(DEV)
    at = lambda off: wide[off:off + M * N].view(M, N)
    if not ops.GEMM_TILE:
        pytest.skip("switched off by PTA_GEMM_TILE=0")
    assert ops.gemm_tile_takes(x, w) and ops.gemm_tile_rule(M, N, K)
    for act in (None, "gelu"):
        for add1, add2 in ((at(1), None), (at(0), at(M * N + 1)), (at(3), at(5))):
            got = ops.mm_rows(x, w, bias, act, add1, add2)
            want = ops.mm_rows(x, w, bias, act, add1.clone(), None if add2 is None else add2.clone())
            assert torch.equal(got, want)


def test_rows_that_share_memory_are_the_librarys():
    """One row seen many times, and rows that overlap: the kernel takes rows that lie a row or more apart."""
    M, N, K = 300, 264, 72
    x, w = _draw(M, N, K, 8)
    flat = x.reshape(-1)
    for rows in (x[:1].expand(M, K), flat.as_strided((M, K), (8, 1))):
        assert not ops.gemm_tile_takes(rows, w)
        got, want = ops.mm_rows(rows, w, None, "gelu"), torch.nn.functional.gelu(rows.double() @ w.double().T)
        assert float((got.double() - want).norm()) <= 2.0 ** -7 * float(want.norm())
