"""Which ranges of K, and which kernel, a pair launch takes: the rule's, and what a table of timed choices has for its shapes (no GPU)."""
import pytest

# (rows of the first matrix, its K, the second's): the rule has one choice up to 32 rows and another from 33 to 64
SHAPES = [(4672, 4544, 18176, 4544), (4544, 18176, 4544, 4544)]


@pytest.fixture
def table():
    """``tuning`` with an empty table active."""
    from pytorch_transformers_amd import tuning

    before = tuning.active()
    tuning.activate(tuning.TuningTable())
    try:
        yield tuning
    finally:
        tuning.activate(before)


def _key(shape):
    return "{}x{},{}x{}".format(*shape)


def _ranges(shape, *rows):
    from pytorch_transformers_amd import ops

    return [ops.gemm_splitk_pair_parts(*shape, M) for M in rows]


@pytest.mark.parametrize("shape", SHAPES)
def test_recorded_ranges_hold_at_every_row_count(table, shape):
    """A table that holds ranges alone, those that the rule has for few rows among them: they are what 33 to 64 rows take too."""
    few, middle = _ranges(shape, 24, 48)
    assert few != middle
    for cut in (few, middle, (1, 1)):
        table.load_tuning({"pair_parts": {_key(shape): [*cut, 1]}})
        assert _ranges(shape, 0, 8, 24, 48, 64) == [cut] * 5
    table.clear_tuning()
    assert _ranges(shape, 24, 48) == [few, middle]


@pytest.mark.parametrize("shape", SHAPES)
def test_ranges_of_33_to_64_rows_are_their_own(table, shape):
    """A table with ranges for both: neither reaches the other's rows, and the table as data brings both back; what the kernel does not
    take is refused."""
    from pytorch_transformers_amd import ops

    lib = ops.load_library()
    first = {"pair_parts": {_key(shape): [2, 1, 1, 4, 2, 2]}, "pair_stationary": {_key(shape): [[0, 0]] * 4}}
    table.load_tuning(first)
    for _ in range(2):
        assert [ops.gemm_splitk_pair_way(*shape, M) for M in (8, 24, 33, 64, 65, 200)] == [(2, 1, 1), (2, 1, 1), (4, 2, 2), (4, 2, 2), (2, 1, 1), (2, 1, 1)]
        kept = table.tuning_table()
        assert kept["pair_parts"] == first["pair_parts"]
        table.clear_tuning()
        table.load_tuning(kept)
    for wrong in ([2, 1, 1, 4, 2, 3], [2, 1, 1, 4, 17, 1], [2, 1, 1, 4]):
        with pytest.raises(ops.KernelError, match="not valid"):
            table.load_tuning({"pair_parts": {_key(shape): wrong}})
    assert lib.pta_gemm_splitk_pair_fix_middle(328, 2112, 200, 4608, 1, 3, 1) == 1, "small matrices have none of their own there"


@pytest.mark.parametrize("times,kept", [([[5.0, 4.0, 3.0]], 2), ([[5.0, 4.9]], 0), ([[5.0, 3.0], [5.0, 5.1]], 0), ([[5.0, 4.5, 3.0], [5.0, 5.0, 5.1]], 1),
                                        ([[5.0]], 0), ([[5.0, 4.0], [5.0, 4.0]], 1)])
def test_the_rule_stays_unless_beaten_at_every_count_of_rows(times, kept):
    from pytorch_transformers_amd import tuning

    assert tuning.pick_way(times, 0.97) == kept


@pytest.mark.parametrize("shape", SHAPES + [(328, 2112, 200, 4608)])
@pytest.mark.parametrize("cls", range(4))
def test_a_class_of_rows_leaves_the_others(table, shape, cls):
    """Where one class of rows is fixed, to the staged kernel or to ranges of the stationary one, the others have what they have without;
    and the staged kernel runs with the rule's ranges of its rows."""
    from pytorch_transformers_amd import ops

    rows = (8, 24, 48, 100)
    plain, fix = _ranges(shape, *rows), ops.load_library().pta_gemm_splitk_pair_fix_stationary
    staged = [plain[i] if i < 2 or (i == 2 and shape in SHAPES) else _ranges(shape, 0)[0] for i in range(4)]
    try:
        for cut, want in (((0, 0), staged[cls]), ((1, 1), (1, 1))):
            assert fix(*shape, cls, *cut) == 0
            assert _ranges(shape, *rows) == [want if i == cls else plain[i] for i in range(4)]
    finally:
        fix(*shape, -1, 0, 0)
    assert _ranges(shape, *rows) == plain


@pytest.mark.parametrize("rows,fix", [(40, "six"), (64, "six"), (64, "stationary"), (8, "stationary")])
def test_whether_attention_rides_is_asked_once_the_pair_is_timed(monkeypatch, rows, fix):
    """Timing may give the pair a launch that carries no attention: the answer has to be the one that holds after it."""
    import types

    import torch
    from pytorch_transformers_amd import ops, tuning

    (N1, K1), (N2, K2) = shapes = (4544, 18176), (4544, 4544)
    lib = ops.load_library()
    empty = lambda *shape: torch.empty(shape, dtype=torch.bfloat16, device="meta")
    x1, w1, w2 = empty(rows, K1), empty(N1, K1), empty(N2, K2)
    late = types.SimpleNamespace(q=empty(rows, 71, 64), k_pool=empty(1, 1, 64, 64))
    cls = [16, 32, 64, 128].index(min(n for n in (16, 32, 64, 128) if n >= rows))

    def timed(*weights):
        assert [tuple(w.shape) for w in weights] == list(shapes)
        if fix == "six":
            assert lib.pta_gemm_splitk_pair_fix_stationary(N1, K1, N2, K2, cls, 0, 0) == 0
            assert lib.pta_gemm_splitk_pair_fix_middle(N1, K1, N2, K2, 3, 1, 4) == 0
        else:
            assert lib.pta_gemm_splitk_pair_fix_stationary(N1, K1, N2, K2, cls, 4, 1) == 0

    before = ops.gemm_splitk_pair_way(N1, K1, N2, K2, rows)
    try:
        assert lib.pta_gemm_splitk_pair_fix(N1, K1, N2, K2, 1, 1, 1) == 0
        assert lib.pta_gemm_splitk_pair_fix_stationary(N1, K1, N2, K2, cls, 0, 0) == 0
        monkeypatch.setattr(tuning, "tune_pair_parts", lambda *weights: None)
        assert ops.gemm_splitk_pair_attn_ok(x1, w1, late, w2)
        monkeypatch.setattr(tuning, "tune_pair_parts", timed)
        assert not ops.gemm_splitk_pair_attn_ok(x1, w1, late, w2)
    finally:
        lib.pta_gemm_splitk_pair_fix(N1, K1, N2, K2, 0, 0, 1)
        lib.pta_gemm_splitk_pair_fix_stationary(N1, K1, N2, K2, -1, 0, 0)
    assert ops.gemm_splitk_pair_way(N1, K1, N2, K2, rows) == before
