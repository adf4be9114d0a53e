"""Prompt tokens per forward: by the weights, unless a class, a model or a pipeline says otherwise."""
import pytest

from umbrella_amd.models.config import LlamaCfg
from umbrella_amd.models.llama import Llama, workspace_rows
from umbrella_amd.parallel import prefill_chunk


def config(awq):
    return LlamaCfg(vocab_size=512, hidden_size=256, intermediate_size=512, num_hidden_layers=4, num_attention_heads=4, num_key_value_heads=2, head_dim=64,
                    rope_theta=10000.0, rope_scaling=None, tie_word_embeddings=False, eos_token_id=[], awq=awq, name="rows")


def model(awq, cls=Llama, **kw):
    return cls("rows", device="cpu", config=config(awq), **kw)


def test_by_the_weights():
    assert model(False).PREFILL_CHUNK == 2048 and model(True).PREFILL_CHUNK == 1024


@pytest.mark.parametrize("awq", [False, True])
@pytest.mark.parametrize("rows", [256, 1024, 4096])
def test_what_a_class_or_a_model_says_stands(awq, rows, monkeypatch):
    class Short(Llama):
        PREFILL_CHUNK = rows
    assert model(awq, Short).PREFILL_CHUNK == rows
    m = model(awq)
    m.PREFILL_CHUNK = rows
    assert m.PREFILL_CHUNK == rows
    monkeypatch.setattr(Llama, "PREFILL_CHUNK", rows)
    assert model(awq).PREFILL_CHUNK == rows


@pytest.mark.parametrize("first,last", [(True, False), (False, False), (False, True)])
def test_a_stage_of_several_sends_messages_that_overlap(first, last):
    """a prompt of 2048 tokens is two messages, so that the stages work side by side; a stage that holds every layer has nobody to send to"""
    m = model(False)
    m.is_first, m.is_last, m.ws_tokens = first, last, 4096
    assert m.PREFILL_CHUNK == 1024 and prefill_chunk(m) == 1024
    m.PREFILL_CHUNK = 512
    assert prefill_chunk(m) == 512
    m = model(False)
    m.is_first = m.is_last = True
    m.ws_tokens = 4096
    assert prefill_chunk(m) == 2048


@pytest.mark.parametrize("awq", [False, True])
def test_no_workspace_for_prompts_that_a_model_cannot_hold(awq):
    short, long = model(awq, max_length=300), model(awq, max_length=8192)
    assert short.max_length == 320 and workspace_rows(short, 64) == 320
    assert workspace_rows(long, 64) == long.PREFILL_CHUNK
    assert workspace_rows(short, 769) == 784 and workspace_rows(long, 4100) == 4112        # a tree's rows are kept, whole tiles of 16
    for m, rows in ((short, 1), (short, 769), (long, 64), (long, 4100)):
        m.ws_tokens = workspace_rows(m, rows)
        assert prefill_chunk(m) <= m.ws_tokens                                             # every message fits the buffers that are made for it
    long.PREFILL_CHUNK = 256
    assert workspace_rows(long, 64) == 256


@pytest.mark.gpu
def test_an_engine_reserves_what_its_models_can_hold():
    import torch
    from helpers import load_golden
    from hip_helpers import static_engine
    eng, _ = static_engine(load_golden(), "cuda:0", torch.float16, self_draft=True, max_length=256)
    for m in (eng.draft_model, eng.target_model):
        assert m.ws_tokens == 256
