"""Memory of captured decode steps: what dropped steps held is given back, and a capture that finds none left tries once more
with torch's cache emptied."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _model():
    from pytorch_transformers_amd import AutoModelForCausalLM, FalconConfig

    cfg = FalconConfig(num_hidden_layers=2, hidden_size=64, num_attention_heads=4, num_kv_heads=2, new_decoder_architecture=True,
                       vocab_size=512, ffn_hidden_size=256, alibi=False, bias=False)
    return AutoModelForCausalLM.from_config(cfg, seed=0, std=0.2, dtype="float32", device="cuda:0")


def test_generating_again_and_again_keeps_no_memory():
    """Each call makes a cache of its own and captures steps in it: the memory torch holds goes up and down, and not up alone."""
    from pytorch_transformers_amd.engine import model as engine

    model, held = _model(), []
    for _ in range(5 * engine.DROPPED_GRAPHS):
        model.generate([[1, 2, 3]], max_new_tokens=4, do_sample=False, eos_token_id=None)
        held.append(torch.cuda.memory_reserved())
    half = len(held) // 2
    assert max(held[half:]) <= max(held[:half])
    assert held[-1] < held[0] + (engine.DROPPED_GRAPHS + 2) * (4 << 20)  # a step's pool here: 2 MiB


def _steps(model, count=4):
    cache = model.new_cache(256, max_slots=2)
    slots = [cache.alloc(), cache.alloc()]
    rows = [model.step(cache, slots, [[5, 6, 7], [8]], "last")]
    rows += [model.step(cache, slots, [[9 + i], [20 + i]], "last") for i in range(count)]
    return torch.stack(rows), cache


def _stateful():
    from pytorch_transformers_amd import AutoModelForCausalLM, PavodraConfig

    mlp = {"kind": "dense", "ff": 128}
    attention = {"heads": 2, "dim": 32, "rot_dim": 16, "vdim": 32, "kv_rank": 64, "scale": 0.15, "rot": {"base": 10000.0, "dims": 16}}
    cfg = PavodraConfig(vocab=512, width=64, layers=[{"type": "latent_attention", "mixer": attention, "mlp": mlp},
                                                     {"type": "mingru", "mixer": {"width": 64}, "mlp": mlp}])
    return AutoModelForCausalLM.from_config(cfg, seed=0, std=0.2, dtype="bfloat16", device="cuda:0")


@pytest.mark.parametrize("make", [_model, _stateful])
@pytest.mark.parametrize("failures", [1, 2])
def test_a_capture_without_memory(monkeypatch, make, failures):
    """The first capture runs out half way: it is taken again.  Where the second attempt runs out too, the step's result stands, as
    the states that layers keep have moved on, and some steps follow without a capture.  Every step's logits are the plain
    steps'."""
    from pytorch_transformers_amd.engine import model as engine

    model = make()
    model.use_graphs = False
    want, _ = _steps(model, 6)
    model.use_graphs = True
    monkeypatch.setattr(engine, "DIRECT_STEPS", 2)
    forward, left, captures = model.forward_tokens, [failures], []

    def short_of_memory(*args):
        out = forward(*args)
        if torch.cuda.is_current_stream_capturing():
            captures.append(1)
            if left[0]:
                left[0] -= 1
                raise torch.cuda.OutOfMemoryError("no memory")
        return out

    monkeypatch.setattr(model, "forward_tokens", short_of_memory)
    got, cache = _steps(model, 6)
    assert torch.equal(got, want) and len(captures) == failures + 1
    assert [(g.graph is not None, g.direct) for g in cache._decode_graphs.values()] == [(True, 0)]
    assert sorted(cache.length(s) for s in range(2)) == [7, 9]


@pytest.mark.parametrize("make", [_model, _stateful])
@pytest.mark.parametrize("failures", [0, 1, 2])
def test_a_shape_captured_before_is_captured_first(monkeypatch, make, failures):
    """In a second cache the step of a known shape is captured and replayed, with no launch of its own; where the capture finds no
    memory twice, the steps are launched directly, and each once: states that layers keep move on by one token a step."""
    from pytorch_transformers_amd.engine import model as engine

    model = make()
    want, _ = _steps(model, 6)
    monkeypatch.setattr(engine, "DIRECT_STEPS", 2)
    forward, left, calls = model.forward_tokens, [failures], []

    def short_of_memory(*args):
        out = forward(*args)
        calls.append(torch.cuda.is_current_stream_capturing())
        if calls[-1] and left[0]:
            left[0] -= 1
            raise torch.cuda.OutOfMemoryError("no memory")
        return out

    monkeypatch.setattr(model, "forward_tokens", short_of_memory)
    got, cache = _steps(model, 6)
    assert torch.equal(got, want)
    # the prompts' step, then captures; with no memory twice: three steps directly, and the next is captured and replayed
    assert calls == [False] + {0: [True], 1: [True, True], 2: [True, True, False, False, False, True]}[failures]
    assert [(g.graph is not None, g.direct) for g in cache._decode_graphs.values()] == [(True, 0)]
    model.tune(table=model.tune(table={}))  # choices may have changed: the next step of the shape sets up what they need
    assert not model._captured_shapes
