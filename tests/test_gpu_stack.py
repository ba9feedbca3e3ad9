"""A prompt's rows by one native call against a call a launch: the same
kernels with the same arguments, so the same bits."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _build():
    from csrc.build import ensure_built
    ensure_built()


def engine(family="llama", hidden=256, hd=64, dtype="bf16", kv="bf16",
           **more):
    import llm_np_cp_amd as L
    from llm_np_cp_amd.io.loader import random_weights
    from llm_np_cp_amd.models.engine import GPUModel

    gemma = family == "gemma2"
    cfg = L.ModelConfig(
        model_type=family, vocab_size=512, hidden_size=hidden,
        intermediate_size=320, num_hidden_layers=3, num_attention_heads=4,
        num_key_value_heads=2, head_dim=hd,
        hidden_act="gelu_pytorch_tanh" if gemma else "silu",
        sliding_window=24 if gemma else None,
        attn_logit_softcapping=50.0 if gemma else None, **more)
    return GPUModel(cfg, random_weights(cfg, seed=3), max_seq=200,
                    max_batch=2, dtype=dtype, kv_dtype=kv)


KINDS = [dict(), dict(kv="fp8"), dict(dtype="fp8"),
         dict(dtype="fp8", kv="fp8", hd=128), dict(dtype="fp4"),
         dict(family="gemma2"), dict(family="gemma2", dtype="fp8", hd=256),
         dict(family="gemma2", dtype="fp4"),
         dict(family="qwen2", attention_bias=True),
         dict(family="qwen2", attention_bias=True, dtype="fp8"),
         dict(family="qwen2", attention_bias=True, dtype="fp4"),
         dict(family="mixtral", num_local_experts=4, num_experts_per_tok=2),
         dict(family="mixtral", num_local_experts=4, num_experts_per_tok=2,
              dtype="fp8"),
         dict(hd=80), dict(hidden=4608), dict(hidden=4608, dtype="fp8")]


# one row, few, the first of many; a second chunk behind the first, in the
# second sequence's cache
@pytest.mark.parametrize("kind", KINDS, ids=lambda k: "-".join(
    str(v) for v in k.values()) or "plain")
def test_one_call_or_one_a_launch(kind):
    m = engine(**kind)
    for chunks in ((1, 2), (16, 1), (17, 70), (130, 5)):
        got = []
        for one in (True, False):
            for t in m.k_cache + m.v_cache:
                t.zero_()
            m._pb, pos, h = 1, 0, []
            rng = np.random.default_rng(sum(chunks))
            for n in chunks:
                ids = rng.integers(0, 512, size=n).astype(np.int32)
                if one:
                    m._read(ids, pos)
                else:
                    m._stack.embed(torch.from_numpy(ids).cuda(), n, pos)
                    m._layers_by_launch(n, keys=pos + n)
                h.append(m.b_h[:n].clone())
                pos += n
            m._pb = 0
            got.append(h + [t[1, :, :pos].clone()
                            for t in m.k_cache + m.v_cache])
        assert m.len_buf.item() == chunks[0]
        for a, b in zip(*got):
            assert torch.isfinite(a.float()).all()
            assert torch.equal(a, b), chunks


# rows of both sequences in a chunk, the second going on behind another
@pytest.mark.parametrize("kind", [k for k in KINDS if k.get("hd") != 80],
                         ids=lambda k: "-".join(
                             str(v) for v in k.values()) or "plain")
@pytest.mark.parametrize("lens", [(3, 4), (40, 60)])
def test_shared_chunk_by_one_call_or_one_a_launch(kind, lens):
    m = engine(**kind)
    rng = np.random.default_rng(sum(lens))
    seqs = [rng.integers(0, 512, size=n).astype(np.int32) for n in lens]
    got = []
    for one in (True, False):
        if not one:
            m._layers_forward = m._layers_by_launch
        for t in m.k_cache + m.v_cache:
            t.zero_()
        cut, h = lens[1] - 2, []
        for segs in ([(1, 0, cut)], [(0, 0, lens[0]), (1, cut, 2)]):
            m._read_pack(segs, seqs)
            h.append(m.b_h[:sum(n for _, _, n in segs)].clone())
        got.append(h + [m.bt_logits32.clone()] +
                   [t[:, :, :max(lens)].clone()
                    for t in m.k_cache + m.v_cache])
    for a, b in zip(*got):
        assert torch.isfinite(a.float()).all()
        assert torch.equal(a, b)
