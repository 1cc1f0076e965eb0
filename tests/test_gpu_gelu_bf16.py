"""The exact GELU of results that are rounded to bfloat16, over every bfloat16 input."""
import numpy as np
import pytest
import torch
from scipy.special import erfc

pytestmark = pytest.mark.gpu

from pytorch_transformers_amd import ops

DEV = "cuda:0"


@pytest.mark.parametrize("cols", [4096, 4095])  # sixteen bytes a thread, one element a thread
def test_every_bfloat16_input_is_rounded_as_from_64_bits(cols):
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    rows = -(-x.numel() // cols)
    y = torch.zeros(rows * cols, dtype=torch.bfloat16)
    y[:x.numel()] = x
    got = ops.epilogue_(y.view(rows, cols).to(DEV), None, "gelu").cpu().view(-1)[:x.numel()].double().numpy()
    xs = x.double().numpy()
    finite = np.isfinite(xs)
    with np.errstate(invalid="ignore"):
        want = np.where(finite, xs * 0.5 * erfc(-xs / np.sqrt(2.0)), 0.0)
    assert got[xs == np.inf] == np.inf and np.isnan(got[xs == -np.inf]).all() and np.isnan(got[np.isnan(xs)]).all()
    assert np.isfinite(got[finite]).all()
    # values that neither 32-bit exponents nor flushed denormals lose: half a unit of eight bits (2^-8 at most), and what the
    # 32-bit arithmetic is off before rounding (under 1e-5 above -13; below that the result is under 1e-37)
    lively = finite & (np.abs(want) > 1e-36)
    off = np.abs(got[lively] - want[lively]) / np.abs(want[lively])
    assert off.max() <= 2.0 ** -8 * (1 + 1e-5) + 1e-5, (off.max(), xs[lively][off.argmax()])
    small = finite & ~lively
    assert np.abs(got[small]).max() <= 2e-36
    # rounded wrongly: none in the arithmetic of numpy, a few where the fast reciprocal is a unit off; the erff form has 188
    nearest = torch.from_numpy(want[lively]).to(torch.bfloat16).double().numpy()
    assert (nearest != got[lively]).sum() <= 16
