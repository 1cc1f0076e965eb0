"""A pair of products is timed with the attention that its launch may carry."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPE = (1024, 16384, 1024, 1024)  # N, K of a block's last matrices, 16 heads of 64 on one KV head


@pytest.fixture
def table():
    from pytorch_transformers_amd import tuning

    before = tuning.active()
    tuning.activate(tuning.TuningTable())
    try:
        yield tuning
    finally:
        tuning.clear_tuning()
        tuning.activate(before)


def _late(M):
    from pytorch_transformers_amd import ops

    draw = lambda *shape: torch.randn(shape, device="cuda").bfloat16()
    i32 = lambda *a: torch.arange(*a, dtype=torch.int32, device="cuda")
    ctx = types.SimpleNamespace(cu_tokens=i32(M + 1), seq_start=torch.full((M,), 20, dtype=torch.int32, device="cuda"), n_seqs=M, n_tokens=M, max_len=21, mean_len=21,
                                is_decode=True, new_tokens=[1] * M, extras={})
    return ops.LateAttention(draw(M, 16, 64), draw(M, 1, 64, 64), draw(M, 1, 64, 64), i32(M).view(M, 1), ctx, None, 0.125, waves=1)


def _timed(ops, tuning, M=8):
    N, K1, _, K2 = SHAPE
    x1, w1, w2 = (torch.randn(s, device="cuda").bfloat16() for s in ((M, K1), (N, K1), (N, K2)))
    late = _late(M)
    with tuning.live_tuning():
        ops.gemm_splitk_pair_attn_ok(x1, w1, late, w2)
    ops.release_flush()
    return lambda rows: bool(ops.load_library().pta_gemm_splitk_pair_attn_ok(*SHAPE, rows, 16, 1, 64))


@pytest.mark.parametrize("gain,carried", [(1e3, True), (-1e3, False)])
def test_ways_that_carry_no_attention_pay_for_it(table, monkeypatch, gain, carried):
    """With a launch of attention that costs a second every class of rows keeps ways that carry it, with one that would save as much none of them
    does: 8 and 32 rows, and 40 and 64, where workgroups of six waves stand against it as well."""
    from pytorch_transformers_amd import ops

    if not table.PAIR_TUNE:
        pytest.skip("timing of pairs is switched off")
    asked = []
    monkeypatch.setattr(table, "ride_gain", lambda copies, late, x1, stream, norm_w: (asked.append(x1.shape[0]), gain)[1])
    carries = _timed(ops, table)
    assert {8, 32, 64} <= set(asked)
    assert [carries(rows) for rows in (8, 32, 40, 64)] == [carried] * 4


def test_what_the_launch_saves_is_timed(table, monkeypatch):
    """As a step is: the attention of as many sequences as rows, both ways with the norm behind them; nothing where it is not carried."""
    from pytorch_transformers_amd import ops

    if not table.PAIR_TUNE:
        pytest.skip("timing of pairs is switched off")
    gains, timed = {}, table.ride_gain
    monkeypatch.setattr(table, "ride_gain", lambda copies, late, x1, *rest: gains.setdefault(x1.shape[0], timed(copies, late, x1, *rest)))
    _timed(ops, table)
    assert gains[128] == 0.0
    for rows in (8, 32):
        assert gains[rows] != 0.0 and abs(gains[rows]) < 0.1  # of microseconds
