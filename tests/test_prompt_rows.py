"""Prompt tokens per forward: by the weights, unless a class, a model or a pipeline says otherwise."""
import pytest

from umbrella_amd.models.config import LlamaCfg
from umbrella_amd.models.llama import Llama


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
