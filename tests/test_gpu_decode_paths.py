"""One row's decode steps through the engine, by each of their ways: a layer's
products in one launch, a launch each where sizes do not let them, and the
same token read as a chunk of one."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def config(family, hidden=256, inter=640, layers=2, experts=0, top=2):
    import llm_np_cp_amd as L
    more = {}
    if family == "gemma2":
        more = dict(attn_logit_softcapping=50.0,
                    final_logit_softcapping=30.0, sliding_window=8)
    if family == "qwen2":
        more = dict(attention_bias=True)
    if experts:
        more = dict(num_local_experts=experts, num_experts_per_tok=top)
    return L.ModelConfig(
        model_type=family, vocab_size=514, hidden_size=hidden,
        intermediate_size=inter, num_hidden_layers=layers,
        num_attention_heads=4, num_key_value_heads=2, head_dim=64,
        hidden_act="gelu_pytorch_tanh" if family == "gemma2" else "silu",
        **more)


def engine(cfg, dtype="bf16", seed=3):
    from llm_np_cp_amd.io.loader import random_weights
    from llm_np_cp_amd.models.engine import GPUModel
    # bf16 values: the router's choice is the oracle's
    w = {k: torch.from_numpy(v).bfloat16().float().numpy()
         for k, v in random_weights(cfg, seed=seed).items()}
    return GPUModel(cfg, dict(w), max_seq=64, dtype=dtype), w


PROMPT = np.arange(5, 16)


def steps(m, tokens=None, n=6):
    """Tokens and logits of n greedy steps behind a prompt, or those of the
    given tokens."""
    m._graph_mode = None
    m.prefill(PROMPT)
    ids, logits = [int(m.decode(1)[0])], []
    for i in range(n):
        if tokens is not None:
            m.next_token.fill_(tokens[i])
        ids.append(int(m.decode(1, use_graph=False,
                                first_from_logits=False)[0]))
        logits.append(m.b_logits.clone())
    return ids, logits


def as_chunks(m, tokens):
    """The logits of the same tokens, each a prompt's chunk of one."""
    cache, _ = m.prefill(PROMPT)
    return [torch.from_numpy(m.forward(np.array([t]), cache,
                                       len(PROMPT) + i)[0].copy()).cuda()
            for i, t in enumerate(tokens)]


# Values are rounded to bf16 some ten times on their way, 2^-9 each at random:
# each way is within 2^-6 of the exact logits.
NEAR = 2.0 ** -5


def off(a, b):
    return ((a - b).norm() / b.norm()).item()


def check_chunks(m, ids, logits):
    """Routed experts beside e4m3 weights read a chunk's rows as e4m3: 2^-4 of
    a value, a mean of many, and a choice of nearly equals may be another."""
    far = sorted(off(a, d) for a, d in zip(logits, as_chunks(m, ids)))
    if m.moe and m.fp8:
        assert far[-2] < 2 * NEAR
    else:
        assert far[-1] < NEAR


@pytest.mark.parametrize("family,dtype,more", [
    *((f, d, {}) for f in ("llama", "gemma2", "qwen2")
      for d in ("bf16", "fp8", "fp4")),
    *(("mixtral", d, dict(experts=e, top=t)) for d in ("bf16", "fp8")
      for e, t in ((4, 2), (8, 2), (3, 1)))])
def test_one_launch_a_layer(family, dtype, more):
    m, _ = engine(config(family, **more), dtype)
    chains = m._chains
    assert len(chains) == 2 and m.launches_only
    ids, logits = steps(m)
    again = steps(m, ids)[1]
    m._chains = None
    single = steps(m, ids)[1]
    for a, b, c in zip(logits, again, single):
        assert torch.equal(a, b)
        assert off(a, c) < NEAR
    check_chunks(m, ids, logits)
    m._chains = chains                        # and its replays
    m._graph_mode = None
    m.prefill(PROMPT)
    assert list(m.decode(7)) == ids


# rows longer than a launch norms, more experts than it chooses from, more of
# them a row: a launch for each product
@pytest.mark.parametrize("family,dtype,more", [
    *((f, d, dict(hidden=4608)) for f in ("llama", "gemma2")
      for d in ("bf16", "fp8", "fp4")),
    *(("mixtral", d, dict(experts=e, top=t)) for d in ("bf16", "fp8")
      for e, t in ((9, 2), (8, 3)))])
def test_a_launch_for_each_product(family, dtype, more):
    from llm_np_cp_amd.models.numpy_ref import NumpyKVCache, NumpyModel
    cfg = config(family, **more)
    m, w = engine(cfg, dtype)
    assert m._chains is None
    ids, logits = steps(m)
    check_chunks(m, ids, logits)
    m.prefill(PROMPT)
    assert list(m.decode(7)) == ids
    if dtype != "bf16":
        return
    ref, cache = NumpyModel(cfg, w), NumpyKVCache(cfg, 64)
    ref.forward(PROMPT, cache, 0)
    for t, z in zip(ids, logits):
        want = torch.from_numpy(np.asarray(
            ref.forward(np.array([t]), cache, cache.seq_len)[-1])).cuda()
        assert off(z, want) < NEAR
