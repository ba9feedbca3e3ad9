"""A group's decode steps through the engine: rows longer than a product norms
by itself, ranges of the history, chunks shorter than the group."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _build():
    from csrc.build import ensure_built
    ensure_built()


def engine(family="llama", hidden=4608, layers=2, **kw):
    import llm_np_cp_amd as L
    from llm_np_cp_amd.io.loader import random_weights
    from llm_np_cp_amd.models.engine import GPUModel

    cfg = L.ModelConfig(
        model_type=family, vocab_size=512, hidden_size=hidden,
        intermediate_size=256, num_hidden_layers=layers,
        num_attention_heads=4, num_key_value_heads=2, head_dim=64,
        hidden_act="gelu_pytorch_tanh" if family == "gemma2" else "silu",
        attn_logit_softcapping=50.0 if family == "gemma2" else None,
        final_logit_softcapping=30.0 if family == "gemma2" else None)
    return GPUModel(cfg, random_weights(cfg, seed=3), max_seq=64,
                    max_batch=4, **kw)


def count(monkeypatch, name):
    from llm_np_cp_amd.ops import hip_ops as ho
    calls, f = [], getattr(ho, name)

    def counted(*a, **k):
        calls.append((a, k))
        return f(*a, **k)
    monkeypatch.setattr(ho, name, counted)
    return calls


def test_rows_that_are_ready_are_not_normed_again(monkeypatch):
    m = engine("gemma2", dtype="fp8")
    m.prefill_batch([[1, 2, 3], [4, 5], [6, 7, 8]])
    calls = count(monkeypatch, "rmsnorm")
    m._layers_forward(3, batch_attn=True)
    # ahead of the first product, then behind each branch
    assert len(calls) == 1 + 2 * 2
