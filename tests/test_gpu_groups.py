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


def engine(family="llama", hidden=4608, layers=2, heads=(4, 2), max_seq=64,
           max_batch=4, more={}, **kw):
    import llm_np_cp_amd as L
    from llm_np_cp_amd.io.loader import random_weights
    from llm_np_cp_amd.models.engine import GPUModel

    cfg = L.ModelConfig(
        model_type=family, vocab_size=512, hidden_size=hidden,
        intermediate_size=256, num_hidden_layers=layers,
        num_attention_heads=heads[0], num_key_value_heads=heads[1],
        head_dim=64,
        hidden_act="gelu_pytorch_tanh" if family == "gemma2" else "silu",
        attn_logit_softcapping=50.0 if family == "gemma2" else None,
        final_logit_softcapping=30.0 if family == "gemma2" else None, **more)
    return GPUModel(cfg, random_weights(cfg, seed=3), max_seq=max_seq,
                    max_batch=max_batch, **kw)


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


# a step's rows go from fp32 to e4m3, however long they are; by way of bf16
# one in fifty takes the other of two e4m3 values (and each scale moves)
@pytest.mark.parametrize("dtype", ["fp8", "fp4"])
@pytest.mark.parametrize("hidden", [4096, 4608])
def test_long_rows_of_a_step_are_rounded_once(hidden, dtype):
    m = engine(hidden=hidden, layers=1, dtype=dtype)
    g = torch.rand(hidden, generator=torch.Generator().manual_seed(1)) + 0.5
    lw = {"wqkv_q": torch.eye(hidden, device="cuda")[:512]
          .to(torch.float8_e4m3fn).view(torch.uint8),
          "wqkv_s": torch.ones(512, device="cuda")}
    m.b_h.normal_(generator=torch.Generator("cuda").manual_seed(2))
    y = torch.zeros(3, 512, dtype=torch.bfloat16, device="cuda")
    # rows of a unit matrix: the product shows what its rows were
    m._rows(lw, "wqkv", m.b_h, y, 3, g=g.cuda(), batch=True)
    x = m.b_h[:3].double()
    x = x * torch.rsqrt(x.pow(2).mean(1, keepdim=True) + 1e-5) \
        * g.cuda().double()
    s = (x.abs().amax(1, keepdim=True) / 448).float()
    q = (x.float() / s).to(torch.float8_e4m3fn).float()[:, :512]
    got = y.float() / s                     # bf16 of q * s: 2^-9 off
    assert ((got - q).abs() > q.abs() * 2.0 ** -6).float().mean() < 0.002


# the rows that are there set the ranges, not those there is room for
@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8"])
def test_ranges_follow_the_active_rows(monkeypatch, kv_dtype):
    m = engine(hidden=256, layers=1, heads=(8, 8), max_seq=2048,
               max_batch=32, kv_dtype=kv_dtype)
    lens = [1900 - 57 * b for b in range(32)]
    for b, n in enumerate(lens):
        m.prefill_row(b, (np.arange(n) * 7 + b) % 512)
    x = torch.randn(32, 256, generator=torch.Generator().manual_seed(1))
    calls, got = count(monkeypatch, "attn_dec"), {}
    for M in (32, 1, 2, 5, 31):
        m.b_h[:M].copy_(x[:M])
        m._layers_forward(M, batch_attn=True)
        got[M] = m.b_att[:M].float()
        assert calls[-1][1]["split"] == min(8, max(1, 32 // M))
        assert not m.bt_attn_cnt.any()
        # sums in another order, bf16 results
        assert (got[M] - got[32][:M]).norm() < 2.0 ** -8 * got[M].norm()


# buffers hold a group's rows where a prompt's chunk is shorter
@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
def test_chunks_shorter_than_the_group(dtype):
    prompts = [[5, 6, 7], [8, 9], [1], [2, 3, 4, 5, 6]] * 5
    ids, h = [], []
    for chunk in (2, 64):
        m = engine(hidden=128, max_batch=20, dtype=dtype, prefill_chunk=chunk)
        ids.append(m.generate_tokens_batch(prompts, 6))
        h.append(m.b_h[:20].float())
        assert m.b_att.shape[0] >= 20 and m.PC == chunk
    assert (h[0] - h[1]).norm() < 0.05 * h[1].norm()
    assert (ids[0] == ids[1]).mean() > 0.9          # ties of close logits


# several prompts in a chunk, one over two chunks, single tokens: the same
# logits as each prompt by itself; a window that ends inside a prompt, norms
# behind the branches, a bias, experts, an e4m3 cache
@pytest.mark.parametrize("dtype", ["bf16", "fp8", "fp4"])
@pytest.mark.parametrize("family,kv,more", [
    ("llama", "bf16", {}), ("llama", "fp8", {}),
    ("gemma2", "bf16", dict(sliding_window=24)),
    ("qwen2", "fp8", dict(attention_bias=True)),
    ("mixtral", "bf16", dict(num_local_experts=4, num_experts_per_tok=2))])
def test_prompts_read_together(family, kv, more, dtype):
    if family == "mixtral" and dtype == "fp4":
        pytest.skip("experts are bf16 or e4m3")
    rng = np.random.default_rng(0)
    prompts = [rng.integers(0, 256, size=n) for n in (5, 40, 1, 33, 65, 2)]
    m = engine(family, hidden=128, max_batch=6, dtype=dtype, kv_dtype=kv,
               prefill_chunk=64, max_seq=80, more=more)
    m.prefill_batch(prompts)
    got = m.bt_logits32[:6].clone()
    for b, p in enumerate(prompts):
        m.prefill_row(b, p)
        want = m.b_logits
        # products in another order, rounded to 8 bits a layer (e4m3 rows: 4)
        bound = 2.0 ** -4 if dtype == "fp8" else 2.0 ** -6
        assert (got[b] - want).norm() < bound * want.norm(), b
    assert m.bt_lens.tolist() == [len(p) for p in prompts]


# more prompts end in a chunk than a launch of heads takes, two, and one by
# itself: a row's logits beside e4m3 weights do not depend on its neighbours
@pytest.mark.parametrize("family", ["llama", "gemma2"])
def test_heads_whatever_the_neighbours(family):
    rng = np.random.default_rng(1)
    prompts = [rng.integers(0, 256, size=2 + b % 3) for b in range(19)]
    full = rng.integers(0, 256, size=64)
    m = engine(family, hidden=128, max_batch=19, dtype="fp8",
               prefill_chunk=64, max_seq=80)
    m.prefill_batch(prompts)
    together = m.bt_logits32[:19].clone()
    for b, p in enumerate(prompts):
        for group in ([p, prompts[0]], [prompts[3], p], [full, p]):
            at = 0 if group[0] is p else 1
            if group[0] is full:              # p in a chunk of its own
                assert [len(c) for c in m._chunks([64, len(p)])] == [1, 1]
            m.prefill_batch(group)
            assert torch.equal(m.bt_logits32[at], together[b]), b
        m.prefill_row(0, p)                   # one row's sums, in their order
        off = (m.b_logits - together[b]).norm() / together[b].norm()
        assert off < 128 * 2.0 ** -23, b
