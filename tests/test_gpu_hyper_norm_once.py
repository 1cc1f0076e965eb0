"""The streams' norm that asks for all of a row at once against the one that walks it."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,width,streams,taps", [(40, 2048, 4, 4), (40, 4096, 2, 3), (40, 1030, 3, 4), (70, 2044, 4, 2), (40, 259, 1, 4)])
def test_a_row_at_once_is_a_row_walked(rows, width, streams, taps, dtype):
    """More than four taps go by the launch that walks a row; with its oldest taps zero it forms the same convolution, so all results have the same
    bits.  Widths that fill the workgroup and that leave threads without features, four and (259) one a thread."""
    from pytorch_transformers_amd import ops

    g = torch.Generator(device="cuda").manual_seed(width + taps)
    draw = lambda *shape: torch.randn(shape, generator=g, device="cuda")
    x, y = draw(rows, streams, width), draw(rows, width).to(dtype)
    mix, out, into, w, conv = draw(streams, streams), draw(streams), draw(streams), draw(width), draw(taps, width)
    tail = draw(rows, (taps - 1) * width)
    more = 5 - taps
    longer = (torch.cat([torch.zeros((more, width), device="cuda"), conv]), torch.cat([draw(rows, more * width), tail], 1))
    ar = torch.arange(rows, dtype=torch.int32, device="cuda")
    ctx = types.SimpleNamespace(token_seq=ar, seq_slot=ar)
    how = dict(y=y, mix=mix, out=out, weights=into, norm=(w, 1.0, 1e-6), want_x=True, want_u=True, want_n=True, want_h=True, ctx=ctx)
    got = ops.hyper_norm(x, streams, dtype, conv=(conv, tail), **how)
    want = ops.hyper_norm(x, streams, dtype, conv=longer, **how)
    for name, a, b in zip(("norm with its convolution", "norm", "sum", "streams"), got, want):
        assert torch.equal(a, b), f"{name}: {int((a != b).sum())} of {a.numel()} differ"
    assert torch.equal(tail, longer[1][:, more * width:])
