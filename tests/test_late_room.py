"""Which pairs of products carry a decode step's attention: those whose second product may wait for it (no GPU)."""
import types

import pytest

# (heads, KV heads, N, K of the first product): a block's last matrices, heads of 64
SIZES = {"7b": (71, 1, 4544, 18176), "40b": (128, 8, 8192, 32768), "4096": (64, 8, 4096, 16384), "1024 wide": (16, 1, 1024, 16384),
         "2048": (32, 8, 2048, 8192), "3072": (48, 1, 3072, 12288), "1024": (16, 1, 1024, 4096), "7b, half": (71, 1, 4544, 9088)}
ROOM = ("7b", "40b", "4096", "1024 wide")


def _pays(size, n_seqs, keys):
    """Of ``late_attention_pays``, asked with tensors' sizes alone."""
    from pytorch_transformers_amd import ops, tuning

    nh, nkv, N, K1 = SIZES[size]
    of = lambda *shape: types.SimpleNamespace(shape=shape)
    late = types.SimpleNamespace(q=of(n_seqs, nh, 64), k_pool=of(9, nkv, 64, 64), ctx=types.SimpleNamespace(n_seqs=n_seqs, max_len=tuning.context_bound(keys), mean_len=keys))
    return ops.late_attention_pays(late, of(N, K1), of(N, nh * 64))


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("n_seqs", [1, 8, 32])
def test_short_contexts(size, n_seqs):
    """The products' own sizes decide: equal workgroups of both wait for nothing, and a launch that ended later for it would cost up to a tenth."""
    assert _pays(size, n_seqs, 60) == _pays(size, n_seqs, 190) == (size in ROOM)


def test_longer_contexts_need_more_room():
    assert [_pays("7b", 8, k) for k in (500, 900, 1900)] == [True, True, True]
    assert [_pays("4096", 8, k) for k in (500, 900, 1900)] == [True, True, False]
    assert [_pays("1024 wide", 8, k) for k in (500, 900, 1900)] == [True, False, False]
    assert [_pays("2048", 8, k) for k in (500, 900, 1900)] == [False, False, False]


def test_ways_that_carry_nothing_have_no_room():
    import ctypes

    from pytorch_transformers_amd import ops

    lib, shapes = ops.load_library(), (1600, 6400, 1600, 1600)
    room = lambda M: [(lib.pta_gemm_splitk_pair_attn_room(*shapes, M, ctypes.byref(r), ctypes.byref(s)), r.value, s.value)
                      for r, s in [(ctypes.c_int(-1), ctypes.c_int(-1))]][0]
    assert lib.pta_gemm_splitk_pair_fix(*shapes, 4, 1, 4) == 0
    try:
        assert lib.pta_gemm_splitk_pair_fix_stationary(*shapes, 2, 0, 0) == 0
        assert room(48) == (0, 0, 0)   # six waves
        rc, rounds, slack = room(8)
        assert rc == 0 and rounds == 1 and slack == 25 - 25  # 100 blocks in four, 25 in one
        assert lib.pta_gemm_splitk_pair_fix(*shapes, 2, 1, 1) == 0
        assert room(48) == (0, 1, 50 - 25)
        assert lib.pta_gemm_splitk_pair_fix_stationary(*shapes, 2, 4, 1) == 0
        assert room(48) == (0, 0, 0)   # stationary activations
    finally:
        lib.pta_gemm_splitk_pair_fix(*shapes, 0, 0, 1)
        lib.pta_gemm_splitk_pair_fix_stationary(*shapes, -1, 0, 0)
    assert lib.pta_gemm_splitk_pair_attn_room(0, 64, 64, 64, 1, ctypes.byref(ctypes.c_int()), ctypes.byref(ctypes.c_int())) != 0


@pytest.mark.parametrize("nh,nkv", [(71, 1), (16, 1), (128, 8), (64, 8), (32, 8), (13, 13), (48, 6)])
def test_short_contexts_are_cut_as_by_a_launch_apart(nh, nkv):
    """Whether attention rides changes no result: up to so many keys a launch apart has one wave on the keys of sixteen heads."""
    from pytorch_transformers_amd import tuning

    for keys in (1, 60, tuning.SHORT_CONTEXT):
        bound = tuning.context_bound(keys)
        assert tuning.short_cut(bound)[2] == 1
        waves = [tuning.late_waves(n, nh, nkv, 64, bound, keys) for n in (1, 2, 4, 5, 8, 16, 33, 64)]
        assert set(waves) <= {0, 1} and waves[0] == 1 and waves == sorted(waves, reverse=True)
