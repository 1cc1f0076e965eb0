"""The sums of squares of the gated norms, to the bit: fused operations in the order of a thread's elements, then the waves' folds."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _fma():
    f = ctypes.CDLL("libm.so.6").fmaf
    f.restype, f.argtypes = ctypes.c_float, [ctypes.c_float] * 3
    return f


def _wave_sum(v):
    """Of 64 32-bit values: halves, quarters and so on added to one another."""
    for o in (32, 16, 8, 4, 2, 1):
        v = v + v[np.arange(64) ^ o]
    return v[0]


def _sum_of_squares(row, threads):
    fma = _fma()
    lanes = np.zeros(threads, dtype=np.float32)
    for t in range(threads):
        s = 0.0
        for v in row[t::threads]:
            s = fma(float(v), float(v), s)
        lanes[t] = s
    total = np.float32(0)
    for w in range(threads // 64):
        total = np.float32(total + _wave_sum(lanes[64 * w:64 * w + 64]))
    return total


def _row_threads(n):  # of a row's workgroup
    return min(1024, max(64, (n // 4 + 63) // 64 * 64))


def _rsqrt(means):
    """The kernel's own 1 / sqrt of each: of a row of one element whose square is nothing, with the number as what is added to its mean."""
    from pytorch_transformers_amd import ops

    tiny, one = torch.tensor([[2.0 ** -80]], device="cuda"), torch.tensor([[float("inf")]], device="cuda")
    return torch.cat([ops.gated_heads(tiny, 1, one, 1, 1, torch.float32, w=torch.tensor([2.0 ** 80], device="cuda"), eps=float(m)) for m in means])


@pytest.mark.parametrize("heads,dv", [(5, 24), (3, 72), (1, 80), (16, 128), (5, 64), (7, 65)])
def test_rows_of_gated_heads(heads, dv):
    from pytorch_transformers_amd import ops

    n, rows, eps = heads * dv, 12, 1e-5
    g = torch.Generator().manual_seed(n)
    x, w = torch.randn((rows, n), generator=g), torch.randn(n, generator=g)
    ss = torch.tensor([_sum_of_squares(r.numpy(), _row_threads(n)) for r in x]).cuda()
    want = x.cuda() * _rsqrt(ss / torch.full_like(ss, n) + eps) * w.cuda()
    got = ops.gated_heads(x.cuda(), dv, torch.full((rows, n), float("inf"), device="cuda"), heads, dv, torch.float32, w=w.cuda(), eps=eps)  # a gate of one
    assert torch.equal(got, want), f"{int((got != want).sum())} of {got.numel()} differ"


@pytest.mark.parametrize("dv", [16, 33, 70, 128, 200, 256, 300])
def test_heads_of_their_own(dv):
    from pytorch_transformers_amd import ops

    heads, rows, eps = 3, 12, 1e-5
    g = torch.Generator().manual_seed(dv)
    x, w = torch.randn((rows, heads * dv), generator=g), torch.randn(dv, generator=g)
    ss = torch.tensor([[_sum_of_squares(h.numpy(), 64) for h in r.view(heads, dv)] for r in x]).cuda()
    want = (x.view(rows, heads, dv).cuda() * (1.0 / torch.sqrt(ss / torch.full_like(ss, dv) + eps))[:, :, None] * w.cuda()).view(rows, -1)
    got = ops.head_norm_gate(x.cuda(), torch.full((rows, heads * dv), float("inf"), device="cuda"), w.cuda(), eps, heads, dv, torch.float32)
    assert torch.equal(got, want), f"{int((got != want).sum())} of {got.numel()} differ"
