"""RMS norm of a 32-bit stream against 64 bits, for rows that can be read four elements at a time and rows that cannot: one and
two chunks a thread, the widest group each kernel takes, groups, gate, residual, picked rows and the sum of streams."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _ops():
    from pytorch_transformers_amd import ops

    ops.load_library()
    return ops


@pytest.mark.parametrize("skew", [0, 1, 2, 4])
@pytest.mark.parametrize("x_wide", [True, False])
@pytest.mark.parametrize("L,groups", [(4, 3), (64, 1), (252, 2), (512, 8), (2048, 1), (4096, 1), (4100, 1), (4228, 2), (8192, 1),
                                      (8196, 1), (2050, 1)])
def test_rmsnorm(L, groups, x_wide, skew):
    """skew: elements that x and the gate start at within wider rows."""
    ops = _ops()
    H, M = L * groups, 5
    g = torch.Generator().manual_seed(L + skew)
    pick = lambda *s: torch.randn(*s, generator=g)
    kind = torch.float32 if x_wide else torch.bfloat16
    x = pick(M, H + skew).to(kind).cuda()[:, skew:]
    gate = pick(M, H + skew).bfloat16().cuda()[:, skew:]
    w, res = pick(H).cuda(), pick(M, H).cuda()
    xd, gd = x.double(), gate.double()

    def want(v, add):
        v = v.view(-1, groups, L)
        n = (v / (v.square().mean(-1, keepdim=True) + 1e-6).sqrt()).reshape(-1, H) * (0.5 + w.double())
        return n if add is None else add.double() + 0.3 * n

    # the sum of L squares in 32 bits, divisions, a root and (gate) an exponential: a few units of the last place each, relative
    # to the norm's own size; the added residual rounds once more
    def check(got, ref, low=False):
        tol = (2.0 ** -24) * (math.sqrt(L) + 32) * ref.abs().clamp(min=1.0) + (2.0 ** -8 * ref.abs() if low else 0)
        assert ((got.double() - ref).abs() <= tol).all()

    how = dict(offset=0.5, groups=groups, want_wide=True)
    narrow, wide = ops.rmsnorm(x, w, 1e-6, torch.bfloat16, **how)
    check(wide, want(xd, None))
    check(narrow, want(xd, None), True)
    narrow, wide = ops.rmsnorm(x, w, 1e-6, torch.bfloat16, gate=gate, residual=res, mult=0.3, **how)
    check(wide, want(xd * gd / (1 + (-gd).exp()), res))
    rows = torch.tensor([4, 0, 2], dtype=torch.int32, device="cuda")
    assert torch.equal(ops.rmsnorm(x, w, 1e-6, torch.bfloat16, gate=gate, residual=res, mult=0.3, rows=rows, **how)[1], wide[rows.long()])
    planes, coef = pick(3, M, H).cuda(), pick(3).cuda()
    before = planes.clone()
    _, mixed = ops.rmsnorm(x, w, 1e-6, torch.bfloat16, gate=gate, residual=res, mult=0.3, mix=(planes, coef, 3), out_wide=planes[2],
                           **how)
    assert torch.equal(planes[2], wide)
    ref = coef[0] * before[0].double() + coef[1] * before[1].double() + coef[2] * wide.double()
    check(mixed, ref)
