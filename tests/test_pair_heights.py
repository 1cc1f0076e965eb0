"""Where a step of 33 to 64 rows runs on workgroups of six waves, by the untimed rule (no GPU)."""
import pytest


@pytest.mark.parametrize("shape", [(6144, 4096, 16384, 4096), (4096, 4096, 4096, 16384), (9216, 8192, 32768, 8192), (4672, 2048, 18176, 2048), (4672, 4544, 18176, 4096)])
@pytest.mark.parametrize("rows", [33, 48, 64])
def test_tiles_that_start_in_places_of_their_own_keep_their_height(shape, rows):
    """Rows of W a multiple of 4 KB long: each tile of rows begins its sums at another place of K, so the height of the tiles is part of the result."""
    from pytorch_transformers_amd import ops

    assert ops.gemm_splitk_pair_way(*shape, rows)[2] in (1, 2, 3)


def test_six_waves_elsewhere():
    from pytorch_transformers_amd import ops

    assert [ops.gemm_splitk_pair_way(4672, 4544, 18176, 4544, rows)[2] for rows in (32, 33, 64)] == [1, 4, 4]
