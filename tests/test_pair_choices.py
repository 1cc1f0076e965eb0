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
