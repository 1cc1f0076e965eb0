"""Timed choices between the ways of a product of many rows: what was timed, or stands in a loaded table, is what runs, and both
sides of a timing do the call's whole work."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _draw(M, N, K, seed=0):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    return r(M, K).bfloat16().cuda(), (0.05 * r(N, K)).bfloat16().cuda()


@pytest.fixture
def ways(monkeypatch):
    """``ops`` with a table of its own, and the names of what products run in, in order: "tile", or rows of a library product."""
    from pytorch_transformers_amd import ops, tuning

    seen, tile, mm = [], ops.gemm_tile_bf16, torch.mm
    monkeypatch.setattr(ops, "gemm_tile_bf16", lambda *a, **k: (seen.append("tile"), tile(*a, **k))[1])
    monkeypatch.setattr(torch, "mm", lambda x, w, **k: (seen.append(x.shape[0]), mm(x, w, **k))[1])
    before = tuning.active()
    tuning.activate(tuning.TuningTable())
    try:
        yield ops, tuning, seen
    finally:
        tuning.activate(before)
        ops.release_flush()


def test_pieces_of_a_table_are_run(ways):
    """A product that the hand-written kernel takes by rule runs in the library's pieces where a table has them, in its kernel where
    that was timed faster, whichever the rule says."""
    ops, tuning, seen = ways
    M, N, K = 1030, 136, 264
    x, w = _draw(M, N, K)
    want = x.double() @ w.double().T
    close = lambda y: float((y.double() - want).norm()) <= 2.0 ** -7 * float(want.norm())
    assert ops.gemm_tile_ok(x, w) and close(ops.mm_rows(x, w)) and seen == ["tile"]
    tuning.load_tuning({"mm_plans": {f"{N},{K},17": [256, 256, 518]}})
    seen.clear()
    assert close(ops.mm_rows(x, w)) and seen == [256, 256, 518]
    for pays in (True, False):
        tuning.load_tuning({"mm_tiles": {f"{N},{K},17,0,0,0": pays}})
        seen.clear()
        assert close(ops.mm_rows(x, w)) and seen == (["tile"] if pays else [256, 256, 518])
    assert tuning.tuning_table()["mm_tiles"] == {f"{N},{K},17,0,0,0": False}


@pytest.mark.parametrize("act,with_bias,adds", [(None, False, 0), ("gelu", True, 0), ("silu", False, 1), (None, False, 2)])
def test_both_ways_are_timed_to_their_end(ways, monkeypatch, act, with_bias, adds):
    """Whichever of the two is faster here, the other one's turn included the bias, the activation and the additions; the choice
    is kept for the shape and the kind of epilogue."""
    ops, tuning, seen = ways
    M, N, K = 300, 520, 264
    x, w = _draw(M, N, K)
    g = torch.Generator().manual_seed(1)
    bias = torch.randn(N, generator=g).cuda() if with_bias else None
    extra = [torch.randn(M, N, generator=g).bfloat16().cuda() for _ in range(adds)] + [None] * (2 - adds)
    passes = []
    epilogue = ops.epilogue_
    monkeypatch.setattr(ops, "epilogue_", lambda y, *a, **k: (passes.append(a), epilogue(y, *a, **k))[1])
    plain = ops.mm_rows(x, w, bias, act, *extra)
    assert not tuning.active().mm_tiles, "nothing is timed unless asked"
    for pick in (0, 1):  # made-up times, after both ways have run
        seen.clear(), passes.clear(), tuning.clear_tuning()

        def times(runs, device):
            got = [run() for run in runs]
            assert len(got) == 2 and all(float((y.float() - plain.float()).norm()) <= 2.0 ** -6 * float(plain.float().norm()) for y in got)
            return [1.0 + (i != pick) for i in range(2)]

        monkeypatch.setattr(tuning, "time_ways_cold", times)
        with ops.live_tuning():
            ops.mm_rows(x, w, bias, act, *extra)
        key = (N, K, 5, ops.ACT_CODES[act], int(with_bias), adds)
        assert tuning.active().mm_tiles == {key: pick == 0}
        assert set(seen[:2]) == {"tile", 300} and seen[2:] == (["tile"] if pick == 0 else [300])
        passes_of = {"tile": int(act == "silu"), 300: int(act is not None or with_bias or adds > 0)}
        assert len(passes) == sum(passes_of[s] for s in seen)
        seen.clear()
        ops.mm_rows(x, w, bias, act, *extra)
        assert seen == (["tile"] if pick == 0 else [300])
