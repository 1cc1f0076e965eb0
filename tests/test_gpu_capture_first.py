"""Which decode steps are captured before they have run: those that ran before, in the same thread and with the same kernels."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _model():
    from pytorch_transformers_amd import AutoModelForCausalLM, FalconConfig

    cfg = FalconConfig(num_hidden_layers=2, hidden_size=256, num_attention_heads=4, num_kv_heads=2, new_decoder_architecture=True,
                       vocab_size=512, ffn_hidden_size=1024, alibi=False, bias=False)
    return AutoModelForCausalLM.from_config(cfg, seed=0, std=0.1, dtype="bfloat16", device="cuda:0")


def _spied(monkeypatch, model):
    """Whether each pass over the model's layers from now on was recorded (True) or ran."""
    calls, forward = [], model.forward_tokens
    monkeypatch.setattr(model, "forward_tokens", lambda *a: (calls.append(torch.cuda.is_current_stream_capturing()), forward(*a))[1])
    return calls


def _step(model):
    cache = model.new_cache(256, max_slots=2)
    slots = [cache.alloc(), cache.alloc()]
    model.step(cache, slots, [[5, 6, 7], [8]], "last")
    return model.step(cache, slots, [[9], [20]], "last")


def test_another_thread_runs_its_first_step(monkeypatch):
    """What libraries set up per thread is not there yet: nothing of a thread's first step of a shape is recorded before it has run."""
    model = _model()
    want = _step(model)
    calls, got = _spied(monkeypatch, model), []
    thread = threading.Thread(target=lambda: got.append(_step(model)))
    thread.start()
    thread.join()
    assert calls == [False, False, True]  # the prompts, the step, and its capture
    assert torch.equal(got[0], want)
    del calls[:]
    assert torch.equal(_step(model), want) and calls == [False, True]  # here it ran before


def test_steps_run_before_they_are_captured_while_choices_are_timed(monkeypatch):
    """Every cut of attention that is timed, and after the timing the first step with what was chosen."""
    from pytorch_transformers_amd import tuning

    model = _model()
    _step(model)
    assert model._captured_shapes
    calls, cuts = _spied(monkeypatch, model), []
    fixed = tuning.set_decode_plan
    monkeypatch.setattr(tuning, "set_decode_plan", lambda key, cut=None: (cuts.append(len(calls)), fixed(key, cut))[1])
    model.tune(prompt_lens=(), batches=(2,), contexts=(700,))
    assert len(cuts) > 2  # the candidates, and what was chosen
    for a, b in zip(cuts, cuts[1:]):
        assert calls[a:b] == [False, True]  # a candidate's step runs and is captured
    assert not model._captured_shapes
    del calls[:]
    _step(model)
    assert calls == [False, False, True]


@pytest.mark.parametrize("change", ["load", "clear", "cut"])
def test_a_choice_that_changes_is_run_first(monkeypatch, change):
    from pytorch_transformers_amd import tuning

    model = _model()
    _step(model)
    if change == "load":
        model.tuning.load({})
    elif change == "clear":
        model.tuning.clear()
    else:
        tuning.set_decode_plan((2, 4, 2, 64, 256, 256), None)
    calls = _spied(monkeypatch, model)
    _step(model)
    assert calls == [False, False, True]
