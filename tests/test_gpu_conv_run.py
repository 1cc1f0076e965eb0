"""The causal convolution of long steps: runs of tokens by four channels a thread, at the edges of a run and of a sequence."""
import pytest
import torch

from pytorch_transformers_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 5])  # five: the kernel of a thread a token and channel
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lengths,channels,before", [([256], 4, 0), ([1, 2, 3, 300, 7, 1], 264, 8), ([255, 8, 1, 40], 1028, 4), ([513], 1028, 1)])
def test_conv_silu_runs(taps, dtype, lengths, channels, before):
    g = torch.Generator().manual_seed(taps * channels)
    M, n = sum(lengths), len(lengths)
    rows = torch.randn(M, before + channels + 8, generator=g).to(dtype)
    x, w, b = rows[:, before:before + channels], torch.randn(channels, taps, generator=g), torch.randn(channels, generator=g)
    tail = torch.randn(n + 2, max(taps - 1, 1) * channels, generator=g)
    slots = torch.randperm(n + 2, generator=g)[:n].int()
    cu = torch.tensor([0] + lengths).cumsum(0).int()
    seq = torch.repeat_interleave(torch.arange(n), torch.tensor(lengths)).int()
    want, size, tail_want = torch.empty(M, channels, dtype=torch.float64), torch.empty(M, channels, dtype=torch.float64), tail.clone()
    for s in range(n):
        old = tail[slots[s]][:(taps - 1) * channels].view(taps - 1, channels)
        line = torch.cat([old, x[cu[s]:cu[s + 1]].float()]).double()
        parts = torch.stack([w[:, k].double() * line[k:k + lengths[s]] for k in range(taps)])
        acc = parts.sum(0) + b.double()
        want[cu[s]:cu[s + 1]], size[cu[s]:cu[s + 1]] = acc / (1 + torch.exp(-acc)), parts.abs().sum(0) + b.double().abs()
        tail_want[slots[s], :(taps - 1) * channels] = line[lengths[s]:].float().flatten()
    d = "cuda:0"
    rows_d, tail_d = rows.to(d), tail.to(d)
    got = ops.conv_silu(rows_d[:, before:before + channels], w.to(d), b.to(d), tail_d, cu.to(d), seq.to(d), slots.to(d))
    # a sum of taps + 1 terms in 32-bit, half an ulp an operation; silu has a slope of at most 1.1; its own two operations and the
    # exponential's few ulps (whose relative error the sigmoid passes on at most)
    bound = 2.0 ** -24 * ((2 * taps + 1) * 1.1 * size + 8 * want.abs()) + 1e-30
    bad = (got.double().cpu() - want).abs() > bound
    assert not bad.any(), (int(bad.sum()), ((got.double().cpu() - want).abs() / bound).max().item())
    assert torch.equal(tail_d.cpu(), tail_want)
