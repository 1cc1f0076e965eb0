"""What the timing of launches counts for each of them (no GPU)."""
import inspect
import re

import pytest


def _launches():
    from pytorch_transformers_amd import ops

    names = set(re.findall(r'_call\(\s*"(pta_\w+)"', inspect.getsource(ops))) - set(ops._HOST_ENTRIES)
    return sorted(n for n in names if re.search(r"gemm_(skinny|splitk|tile|normed|f32)|attn|scan|ssm|delta|linear_state", n))


def test_no_launch_of_a_product_or_a_state_counts_for_nothing(monkeypatch):
    """With every size 2: a product reads its matrices, a recurrence its state or its rows, attention what the caller says."""
    from pytorch_transformers_amd import ops

    monkeypatch.setattr(ops, "timing_hint", {"attn_bytes": 1, "attn_flops": 1, "rows": 1})
    launches = _launches()
    assert {"pta_gemm_splitk_pair_attn", "pta_ssm_step", "pta_gemm_f32_pair", "pta_gemm_splitk_bf16"} <= set(launches)
    free = {n for n in launches if ops._entry_cost(n, [2] * 48)[0] <= 0}
    assert not free, sorted(free)


def test_a_pair_that_carries_attention(monkeypatch):
    """Is its two matrices and the attention."""
    from pytorch_transformers_amd import ops

    monkeypatch.setattr(ops, "timing_hint", {"attn_bytes": 1000, "attn_flops": 500})
    args = [0] * 28
    args[3], args[4], args[8], args[9], args[10] = 4544, 18176, 4544, 4544, 8
    matrices = 4544 * (18176 + 4544)
    assert ops._entry_cost("pta_gemm_splitk_pair_attn", args) == (2.0 * matrices + 1000, 2.0 * 8 * matrices + 500)


@pytest.mark.parametrize("code,size", [(0, 4.0), (1, 2.0)])
def test_a_step_of_the_state_space_mixer(code, size):
    from pytorch_transformers_amd import ops

    args = [0] * 24
    args[17:23] = [8, 64, 128, 8, 4, code]
    state, channels = 64 * 64 * 128, 64 * 64 + 2 * 8 * 128
    nbytes, flops = ops._entry_cost("pta_ssm_step", args)
    assert nbytes == 8 * (8.0 * (state + 3 * channels) + size * (2 * 64 * 64 + channels + 64))
    assert flops == 4.0 * 8 * state
