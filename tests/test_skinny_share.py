"""How the few-row products' launches tell a workgroup which rows of W are its own (no GPU)."""
import ctypes

import pytest


def _share(items, groups, j):
    from pytorch_transformers_amd import ops

    begin, end = ctypes.c_int(-1), ctypes.c_int(-1)
    if ops.load_library().pta_gemm_skinny_share(items, groups, j, ctypes.byref(begin), ctypes.byref(end)):
        return None
    return begin.value, end.value


@pytest.mark.parametrize("rows", [1, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("groups", [1, 2, 64, 255, 256, 257, 512])
def test_every_row_is_one_workgroups(rows, groups):
    """Full workgroups of every height (64 rows for each of 64, 256, 512 ..), one row fewer, and an uneven rest."""
    for items in {rows * groups, rows * groups - 1, rows * groups - groups // 2, (rows - 1) * groups + 1}:
        if items < groups:
            continue
        shares = [_share(items, groups, j) for j in range(groups)]
        assert shares[0][0] == 0 and shares[-1][1] == items
        assert all(a[1] == b[0] for a, b in zip(shares, shares[1:]))
        assert {b - a for a, b in shares} <= {items // groups, items // groups + 1}


@pytest.mark.parametrize("items,groups", [(2 ** 31 - 64, 2 ** 25 - 1), (2 ** 31 - 1, 2 ** 25), (2 ** 31 - 1, 2 ** 26 - 1)])
def test_the_most_workgroups(items, groups):
    assert _share(items, groups, 0) == (0, items // groups + (items % groups > 0))
    assert _share(items, groups, groups - 1) == (items - items // groups, items)


def test_more_rows_than_a_workgroup_has_are_refused():
    assert _share(65 * 256, 256, 0) is None and _share(64 * 256 + 1, 256, 0) is None
