"""Whether a pair of 32-bit products has a launch is asked four times in a prompt of two layers: the number of rows and the type answer it alone."""
from types import SimpleNamespace

import pytest
import torch

from pytorch_transformers_amd import ops


@pytest.mark.parametrize("rows,dtype", [(17, torch.float32), (2048, torch.float32), (8, torch.bfloat16)])
def test_rows_and_type_alone_refuse(rows, dtype):
    assert not ops.gemm_f32_pair_ok(SimpleNamespace(dtype=dtype, shape=(rows, 64)), None, None, None)
