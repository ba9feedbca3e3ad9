"""The rows that the chunks of a long prompt are given."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def engine(family="llama", hidden=2304, dtype="bf16", max_batch=1, **more):
    import llm_np_cp_amd as L
    from llm_np_cp_amd.io.loader import random_weights
    from llm_np_cp_amd.models.engine import GPUModel

    gemma = family == "gemma2"
    cfg = L.ModelConfig(
        model_type=family, vocab_size=512, hidden_size=hidden,
        intermediate_size=9216, num_hidden_layers=1, num_attention_heads=8,
        num_key_value_heads=4, head_dim=256,
        hidden_act="gelu_pytorch_tanh" if gemma else "silu", **more)
    return GPUModel(cfg, random_weights(cfg, seed=3), max_seq=4200,
                    dtype=dtype, max_batch=max_batch)


@pytest.mark.parametrize("kind", [
    dict(), dict(family="gemma2"), dict(hidden=2048), dict(dtype="fp4"),
    dict(dtype="fp8"),
    dict(family="mixtral", num_local_experts=4, num_experts_per_tok=2)])
def test_as_many_chunks_of_whole_tiles(kind):
    m = engine(**kind)
    some = 0
    for most in (2048, 1000, 128, 1):
        for n in (1, most, most + 1, most + most // 2, 2 * most,
                  2 * most + 903, 5 * most - 7):
            rows = m._stack.chunk_rows(n, most)
            assert rows == most or (rows < most and rows % 128 == 0 and
                                    -(-n // rows) == -(-n // most))
            assert rows == most or n > most
            some += rows < most
    still = kind.get("dtype") == "fp8" or "num_local_experts" in kind
    assert not (still and some)
    if kind in ({}, dict(family="gemma2")):
        assert m._stack.chunk_rows(3000, 2048) == 1792


@pytest.mark.parametrize("kind", [dict(), dict(dtype="fp4")])
def test_the_same_prompt(kind):
    """By chunks of either number of rows: bf16 results of sums in another
    order, 2^-8 of them and what one layer and the head add to that."""
    m = engine(**kind)
    ids = np.arange(3001) * 7 % 512
    got = []
    for rows in (m._chunk_rows, lambda n: 2048, lambda n: 1536):
        m._chunk_rows = rows
        _, logits = m.prefill(ids)
        got.append(logits.copy())
        assert m.len_buf.item() == 3001
    for other in got[1:]:
        assert np.linalg.norm(other - got[0]) < \
            2.0 ** -6 * np.linalg.norm(got[0])


@pytest.mark.parametrize("kind", [dict(), dict(dtype="fp4"),
                                  dict(dtype="fp8")])
def test_the_same_by_each_entry_point(kind):
    """A long prompt alone: prefill, a row of a pool, a group of one."""
    m = engine(max_batch=2, **kind)
    ids = np.arange(3001) * 7 % 512
    _, want = m.prefill(ids)
    want = want[0].copy()
    m.prefill_batch([ids])
    assert np.array_equal(m.bt_logits32[0].cpu().numpy(), want)
    m.prefill_row(1, ids)
    assert np.array_equal(m.b_logits.cpu().numpy(), want)
