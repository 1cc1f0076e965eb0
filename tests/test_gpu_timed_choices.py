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

    if not (ops.GEMM_TILE and tuning.MM_CHUNKS):
        pytest.skip("switched off by PTA_GEMM_TILE=0 or PTA_MM_CHUNKS=0")
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

    def runs():
        seen.clear()
        y = ops.mm_rows(x, w)
        assert float((y.double() - want).norm()) <= 2.0 ** -7 * float(want.norm())
        return list(seen)

    assert runs() == ["tile"]
    tuning.load_tuning({"mm_plans": {f"{N},{K},17": [256, 256, 518]}})
    assert runs() == [256, 256, 518]
    for pays in (True, False):
        tuning.load_tuning({"mm_tiles": {f"{N},{K},17,0,0,0": pays}})
        assert runs() == (["tile"] if pays else [256, 256, 518])
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


@pytest.mark.parametrize("act,with_bias", [("gelu", False), (None, True), (None, False)])
def test_joined_matrices_are_timed_with_what_follows_them(ways, monkeypatch, act, with_bias):
    """Two matrices of one input, in one product or each in its own: on either side bias and activation are part of what is
    timed, and the answer counts for that epilogue; a table that knows the shape alone still holds."""
    from pytorch_transformers_amd.parts import Linear

    ops, tuning, _ = ways
    if not tuning.MM_JOIN:
        pytest.skip("switched off by PTA_MM_JOIN=0")
    M, N1, N2, K = 600, 72, 136, 200
    g = torch.Generator().manual_seed(2)
    first, second = Linear("a", K, N1, False), Linear("b", K, N2, False)
    first.weight, second.weight = ((0.05 * torch.randn(n, K, generator=g)).bfloat16().cuda() for n in (N1, N2))
    first.bias = second.bias = first.joined = second.joined = None
    if with_bias:
        second.bias = torch.randn(N2, generator=g).cuda()
    assert Linear.join(first, second)
    x = torch.randn(M, K, generator=g).bfloat16().cuda()
    work = []  # (rows of the matrix, whether its epilogue came with it), and the passes
    mm_rows, epilogue = ops.mm_rows, ops.epilogue_
    monkeypatch.setattr(ops, "mm_rows", lambda x, w, b=None, a=None, *r: (work.append((w.shape[0], a is not None or b is not None)), mm_rows(x, w, b, a, *r))[1])
    monkeypatch.setattr(ops, "epilogue_", lambda y, *a: (work.append((y.shape[1], "pass")), epilogue(y, *a))[1])
    monkeypatch.setattr(tuning, "tile_pays", lambda *a: True)  # (the products' own choice is another test's)
    with ops.live_tuning():
        both = Linear.pair(first, x, {}, second, x, {"act": act})
    ep = act is not None or with_bias
    joined, apart = [(N1 + N2, False)] + [(N2, "pass")] * ep, [(N1, False), (N2, ep)]
    assert work[:5 * len(joined + apart)] == (joined + apart) * 5  # one run each before the timing, four in it
    key = (N1, N2, K, 10) + ((0, 0, ops.ACT_CODES[act], int(with_bias)) if ep else ())
    pays = tuning.active().mm_joined.get(key)
    assert list(tuning.active().mm_joined) == [key] and (both is not None) == pays
    # a loaded table: by the whole key, or by the shape alone as older tables have it
    for k in (key, key[:4]):
        for pays in (True, False):
            tuning.clear_tuning()
            tuning.load_tuning({"mm_joined": {",".join(map(str, k)): pays}})
            both = Linear.pair(first, x, {}, second, x, {"act": act})
            assert (both is not None) == pays
            if pays:
                want = x.double() @ second.weight.double().T + (second.bias.double() if with_bias else 0.0)
                want = torch.nn.functional.gelu(want) if act else want
                assert float((both[1].double() - want).norm()) <= 2.0 ** -7 * float(want.norm())


def test_ranges_of_k_are_timed_to_their_end(ways, monkeypatch):
    """The product over ranges of K and the one in one, each with its bias, activation and additions; and the one in one is
    whichever ``whole_rows`` is."""
    ops, tuning, _ = ways
    if not ops.MM_KSPLIT:
        pytest.skip("switched off by PTA_MM_KSPLIT=0")
    M, N, K = 300, 136, 640
    x, w = _draw(M, N, K)
    g = torch.Generator().manual_seed(3)
    bias, add = torch.randn(N, generator=g).cuda(), torch.randn(M, N, generator=g).bfloat16().cuda()
    want = torch.nn.functional.gelu(x.double() @ w.double().T + bias.double()) + add.double()
    monkeypatch.setattr(tuning, "tile_pays", lambda *a: True)
    for pick in range(3):
        tuning.clear_tuning()

        def times(runs, device):
            got = [run() for run in runs]
            assert len(got) == 3 and all(float((y.double() - want).norm()) <= 2.0 ** -7 * float(want.norm()) for y in got)
            return [1.0 - 0.5 * (i == pick) for i in range(3)]

        monkeypatch.setattr(tuning, "time_ways_cold", times)
        with ops.live_tuning():
            assert (ops.library_mm_ksplit(x, w, bias, "gelu", add) is None) == (pick == 0)
        assert tuning.active().mm_ksplit == {(N, K, 5): (1, 2, 4)[pick]}
