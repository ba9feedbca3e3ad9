"""Garupel on the GPU against the plain oracle (float64): every mechanism
alone, any cut of the tokens, mixed batches, reused pages and slots, keys
and inputs that stand out, long decoding and the framework's generation
paths.

Caches and states start filled with NaN, so reading a position or a state
that the sequence has not written fails the comparison.
"""

import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from garupel_cases import (attention, config, default, greedy, lightning, rel,
                           rglru, save, tokens, weights, worst)
from garupel_oracle import Oracle
from layered_gpu import EXACT, ROUNDED, cut, engine, entry, run

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ---------------------------------------------------------------- kernels

def _dev(a, dtype=torch.float32):
    return torch.from_numpy(np.asarray(a, np.float32)).to("cuda", dtype)


def _np(t):
    return t.double().cpu().numpy()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [8, 88, 513, 2048, 2113, 5000])
def test_staging_of_rows(dtype, width):
    """Post norm + addition + embedding + norm (+ gate) of rows, in place
    and beside, alone and inside a one-row projection."""
    from llm_np_cp_amd.ops import hybrid_ops as hy

    rng = np.random.default_rng(width)
    n, Kp, N, eps = 5, -(-width // 64) * 64, 53, 1e-5
    x, y, x0, gate = (rng.standard_normal((n, width)) * s
                      for s in (3, 0.2, 1, 2))
    g, gb = rng.standard_normal(width) + 1, rng.standard_normal(width)
    rms = lambda a: a / np.sqrt((a * a).mean(-1, keepdims=True) + eps)
    X, Y, X0, GT, G, GB = map(_dev, (x, y, x0, gate, g, gb))
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    h = torch.full((n, Kp), float("nan"), dtype=dtype, device="cuda")
    for xadd in (None, X0):
        v = x + rms(y) * gb + (x0 if xadd is not None else 0)
        out = torch.full((n, width), float("nan"), device="cuda")
        hy.norm_rows(X, G, h, n, width, Kp, eps, y=Y, gb=GB, xadd=xadd,
                     xout=out)
        assert rel(_np(h[:, :width]), rms(v) * g) < tol
        assert (h[:, width:] == 0).all() and rel(_np(out), v) < 1e-5
        inplace = X.clone()
        hy.norm_rows(inplace, None, None, n, width, width, eps, y=Y, gb=GB,
                     xadd=xadd, xout=inplace)
        assert torch.equal(inplace, out)
    hy.norm_rows(X, G, h, n, width, Kp, eps, gate=GT, ldg=width)
    assert rel(_np(h[:, :width]), rms(x) * g / (1 + np.exp(-gate))) < tol

    W = torch.zeros(N, Kp, dtype=dtype, device="cuda")
    W[:, :width] = _dev(rng.standard_normal((N, width)) / width ** .5, dtype)
    Wr, bias = _np(W[:, :width]), rng.standard_normal(N)
    v = x + rms(y) * gb + x0
    z = rms(v) * g @ Wr.T
    out = torch.full((width + 1,), 9.0, device="cuda")
    got = torch.full((N + 1,), 7.0, device="cuda")
    hy.lin_row(W, X, got, width, eps, g=G, res=Y, gb=GB, xadd=X0, xout=out,
               bias=_dev(bias))
    assert rel(_np(got[:N]), z[0] + bias) < tol and got[N] == 7.0
    assert rel(_np(out[:width]), v[0]) < 1e-5 and out[width] == 9.0
    sq = torch.full((N,), float("nan"), dtype=dtype, device="cuda")
    rows = torch.tensor([3], dtype=torch.int32, device="cuda")
    hy.lin_row(W, X, sq, width, eps, g=G, res=Y, gb=GB, xadd=X0, rows=rows,
               epi=hy.EPI_RELU2)
    assert rel(_np(sq), np.maximum(z[3], 0) ** 2) < tol
    hy.lin_row(W, X, got, width, eps, g=G, gate=GT, ldg=width)
    assert rel(_np(got[:N]),
               rms(x[0]) * g / (1 + np.exp(-gate[0])) @ Wr.T) < tol
    hy.lin_row(W, None, got, 0, 0.0, hin=h)
    assert rel(_np(got[:N]), _np(h[0]) @ _np(W).T) < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M, N, K", [(2, 40, 64), (17, 70, 128), (64, 33, 64),
                                     (200, 257, 192), (2500, 2049, 64),
                                     (2500, 2433, 64)])
def test_gemm_bias_and_squared_relu(dtype, M, N, K):
    from llm_np_cp_amd.ops import hybrid_ops as hy

    g = torch.Generator(device="cuda").manual_seed(M)
    R = lambda *s: torch.randn(*s, device="cuda", generator=g)
    X, W, b = R(M, K).to(dtype), (R(N, K) / K ** 0.5).to(dtype), R(N)
    ref = _np(X) @ _np(W).T
    Y = torch.empty(M, N, device="cuda")
    hy.gemm_rows(X, W, Y, M, K, N, hy.EPI_F32, bias=b)
    assert rel(_np(Y), ref + _np(b)) < 1e-5
    A = torch.empty(M, N, dtype=dtype, device="cuda")
    hy.gemm_rows(X, W, A, M, K, N, hy.EPI_RELU2)
    assert rel(_np(A), np.maximum(ref, 0) ** 2) < (
        1e-5 if dtype == torch.float32 else 5e-3)


def test_launchers_refuse_bad_shapes():
    from llm_np_cp_amd.ops import hybrid_ops as hy

    t = torch.zeros(64, 64, device="cuda")
    with pytest.raises(RuntimeError):
        hy.norm_rows(t, None, None, 2, 64, 64, 1e-5)      # nothing to write
    with pytest.raises(RuntimeError):                     # in place, one row
        hy.lin_row(t, t, torch.zeros(64, device="cuda"), 64, 1e-5, g=t,
                   res=t, gb=t, xout=t)
    a = hy.GqaArgs().put(H=6, G=4, d=8, vd=8, DP=64, VP=64, ldo=64, rows=1,
                         NS=2)
    with pytest.raises(RuntimeError):
        hy.gqa_token(1, a)
    with pytest.raises(RuntimeError):
        hy.rglru_step(1, hy.RglruArgs().put(rows=1, C=10, nb=3, bw=3, KP=64,
                                            taps=1, ldo=64))
    with pytest.raises(RuntimeError):
        hy.lightning_step(hy.LightningArgs().put(rows=1, H=1, d=8, vd=65,
                                                 nvt=1))


# the new token first, last and amid a share's 32 keys, a page, 128 keys; in a
# share's first group and in a later one; a cache that holds anything where no
# token has written
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H, G, d, vd", [(6, 2, 40, 72), (17, 1, 64, 30),
                                         (4, 4, 130, 20)])
@pytest.mark.parametrize("pos, NS", [([0, 31, 32], 1), ([63, 64, 127], 2),
                                     ([128, 500, 255], 2), ([300, 1, 17], 5)])
def test_new_token_among_keys_read_before_it(dtype, H, G, d, vd, pos, NS):
    from llm_np_cp_amd.ops import hybrid_ops as hy

    g = torch.Generator(device="cuda").manual_seed(d)
    R = lambda *s: torch.randn(*s, device="cuda", generator=g)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
    DP, VP = (256, 256) if d > 128 else (64, 64 if vd <= 64 else 128)
    n, per, R_ = len(pos), max(pos) // 64 + 1, H // G
    ov = H * d + G * d
    P, qn, kn = R(n, ov + G * vd), R(H * d), R(G * d)
    table = i32(*torch.randperm(n * per).tolist()).view(n, per)
    K = torch.full((n * per, G, 64, DP), float("nan"), device="cuda",
                   dtype=dtype)
    V = torch.full((n * per, G, VP, 64), float("nan"), device="cuda",
                   dtype=dtype)
    K[..., d:] = 0
    V[:, :, vd:] = 0
    norm = lambda x: x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5)
    q = (norm(P[:, :H * d]) * qn).to(dtype).double().view(n, H, d)
    k1 = (norm(P[:, H * d:ov]) * kn).to(dtype).view(n, G, d)
    v1 = P[:, ov:].to(dtype).view(n, G, vd)
    want = torch.zeros(n, H, vd, dtype=torch.float64)
    for r in range(n):
        ks, vs = R(pos[r], G, d).to(dtype), R(pos[r], G, vd).to(dtype)
        for j in range(pos[r]):
            at, o = int(table[r, j // 64]), j % 64
            K[at, :, o, :d] = ks[j]
            V[at, :, :vd, (o & 32) | ((o >> 2) & 3) << 3 | ((o >> 4) & 1) << 2
              | (o & 3)] = vs[j]
        ks, vs = torch.cat([ks, k1[r:r + 1]]), torch.cat([vs, v1[r:r + 1]])
        for h in range(H):
            s = ks[:, h // R_].double() @ q[r, h] * d ** -0.5
            want[r, h] = (s.softmax(0) @ vs[:, h // R_].double()).cpu()
    part = torch.zeros(NS, n * H, VP, device="cuda")
    ml = torch.zeros(NS, n * H, 2, device="cuda")
    out = torch.zeros(n, H * vd, device="cuda", dtype=dtype)
    f32, slot, at = int(dtype == torch.float32), i32(*range(n)), i32(*pos)
    a = hy.GqaArgs().put(
        P=P, qnorm=qn, knorm=kn, slot=slot, pos=at,
        table=table, K=K, V=V, part=part, ml=ml, o=out, ldp=P.shape[1], oq=0,
        ok=H * d, ov=ov, og=-1, H=H, G=G, d=d, vd=vd, DP=DP, VP=VP,
        ldo=H * vd, ldt=per, rows=n, rbase=0, NS=NS, eps=1e-5,
        scale=d ** -0.5)
    hy.gqa_token(f32, a)
    hy.gqa_merge(f32, a)
    # bf16: keys and queries a unit apart where the norm's sum has another
    # order (2^-8 of some), probabilities and results rounded (2^-9 each)
    assert rel(_np(out), want.view(n, -1).numpy()) < (
        1e-5 if f32 else 2.0 ** -7)
    for r in range(n):
        o = pos[r] % 64
        new = K[table[r, pos[r] // 64], :, o, :d]
        assert rel(_np(new), _np(k1[r])) < (1e-5 if f32 else 2.0 ** -8)


# -------------------------------------------------------- mechanisms alone

def check_alone(cfg, n=150, seed=0, cuts=None):
    w, t = weights(cfg, seed), tokens(cfg, n)
    want, _ = Oracle(cfg, w).run(t)
    cuts = cuts or ([n], [1] * 70 + [2, n - 72], cut(n, [64, 1, 65, 20]))
    m = engine(cfg, w)
    for c in cuts:
        assert worst(run(m, t, c), want) < EXACT, c
    m = engine(cfg, w, "bf16")
    for c in cuts:
        assert rel(run(m, t, c), want) < ROUNDED, c


ATTENTIONS = [attention(), attention(1, 1, 8, 8, every=1),
              attention(4, 4, 64, 64, every=50), attention(8, 2, 40, 72),
              attention(3, 1, 65, 30, 0.2), attention(10, 5, 128, 128),
              attention(17, 1, 16, 24), attention(40, 2, 12, 20, coef=0.0),
              attention(2, 1, 130, 200), attention(6, 2, 256, 16),
              attention(5, 5, 33, 129, 0.02, -0.05, 9)]


@pytest.mark.parametrize("k", range(len(ATTENTIONS)))
def test_attention_alone(k):
    check_alone(config([(ATTENTIONS[k], None)]), seed=k)


RGLRUS = [rglru(), rglru(24, 1, 1), rglru(64, 1, 4), rglru(130, 2, 2),
          rglru(260, 2, 3), rglru(96, 16, 4), rglru(150, 1, 6),
          rglru(40, 40, 9), rglru(512, 4, 5)]


@pytest.mark.parametrize("k", range(len(RGLRUS)))
def test_rglru_alone(k):
    check_alone(config([(RGLRUS[k], None)]), n=200, seed=k, cuts=(
        [200], [1] * 70 + [2, 128], [63, 1, 65, 64, 7], cut(200, [2]),
        cut(200, [3, 1, 2, 70])))


LIGHTNINGS = [lightning(), lightning(1, 4, 4), lightning(2, 64, 64),
              lightning(3, 100, 30), lightning(7, 16, 130),
              lightning(1, 200, 200), lightning(2, 24, 40, [1.0, 0.0])]


@pytest.mark.parametrize("k", range(len(LIGHTNINGS)))
def test_lightning_alone(k):
    check_alone(config([(LIGHTNINGS[k], None)]), n=200, seed=k, cuts=(
        [200], [1] * 70 + [2, 128], [63, 1, 65, 64, 7]))


@pytest.mark.parametrize("ff", [1, 40, 64, 200])
@pytest.mark.parametrize("T", [1, 4, 23, 90])
def test_dense_alone(ff, T):
    """A mixer that writes nothing: its post norm leaves 0 (plus nothing)."""
    cfg = config([(attention(2, 1), ff)], width=72)
    w = weights(cfg)
    w["l0.mix.o"] *= 0
    t = tokens(cfg, T)
    want, _ = Oracle(cfg, w).run(t)
    m = engine(cfg, w)
    assert worst(run(m, t), want) < EXACT
    assert worst(run(m, t, [1] * T), want) < EXACT


@pytest.mark.parametrize("loop", [(0, 1, 1), (0, 2, 3), (1, 2, 2), (1, 3, 4),
                                  (0, 3, 2)])
def test_loop_alone(loop):
    """Without the sublayers only the additions of the embedding are left."""
    cfg = config([(attention(2, 1), None), (rglru(), None),
                  (lightning(), 40)], loop=loop)
    w, t = weights(cfg), tokens(cfg, 9)
    w["final.norm"][:] = 1
    for k in w:
        if k.endswith(("norm1b", "norm2b")):
            w[k] *= 0
    want, _ = Oracle(cfg, w).run(t)
    m = engine(cfg, w)
    x, hidden = m.forward_full(t, return_hidden_states=True)
    assert worst(x, want) < EXACT
    assert rel(hidden[-1], loop[2] * w["embed"][t]) < 1e-5
    assert worst(run(m, t, [1] * 9), want) < EXACT


def test_loop_passes_keep_their_own_cache():
    cfg = config([(attention(), None), (rglru(), 40), (lightning(), None)],
                 loop=(0, 3, 3))
    w, t = weights(cfg), tokens(cfg, 80)
    want, _ = Oracle(cfg, w).run(t)
    m = engine(cfg, w)
    assert len(m.caches) == 9
    assert worst(run(m, t), want) < EXACT
    assert worst(run(m, t, [1] * 80), want) < EXACT


@pytest.mark.parametrize("kw", [dict(width=64, vocab=64), dict(width=130),
                                dict(eps=0.3), dict(vocab=1001),
                                dict(width=520)])
def test_stack_constants(kw):
    cfg = config([(attention(), 50), (rglru(), None), (lightning(), 100)],
                 **kw)
    w, t = weights(cfg), tokens(cfg, 21)
    want, _ = Oracle(cfg, w).run(t)
    m = engine(cfg, w)
    assert worst(run(m, t), want) < EXACT
    assert worst(run(m, t, [1] * 21), want) < EXACT


@pytest.mark.parametrize("lam, bias", [(-12.0, 0.0), (9.0, 6.0), (-3.0, -9.0)])
def test_rglru_at_its_extremes(lam, bias):
    """Decays of almost 1 (the root of 1 - a^2 cancels), of almost 0, and
    closed gates."""
    cfg = config([(rglru(48, 3, 3), None)])
    w, t = weights(cfg), tokens(cfg, 190)
    w["l0.mix.lam"][:] = lam
    w["l0.mix.ra.b"][:] = bias
    want, _ = Oracle(cfg, w).run(t)
    m = engine(cfg, w)
    for cuts in ([190], [1] * 190, cut(190, [5, 1, 70, 2])):
        assert worst(run(m, t, cuts), want) < EXACT


# ------------------------------------------------------------- whole model

@pytest.fixture(scope="module")
def model():
    cfg = default()
    w = weights(cfg)
    t = tokens(cfg, 300)
    return cfg, w, t, Oracle(cfg, w).run(t)[0]


def test_residual_after_every_layer_run(model):
    cfg, w, t, _ = model
    trace = []
    logits, _ = Oracle(cfg, w).run(t[:30], trace=trace)
    m = engine(cfg, w)
    got, hidden = m.forward_full(t[:30], return_hidden_states=True)
    assert len(hidden) == len(trace) + 1
    for a, b in zip(hidden[1:], trace):
        assert worst(a, b) < EXACT
    assert worst(got, logits) < EXACT


@pytest.mark.parametrize("sizes", [[300], [1], [2], [3, 1], [5, 2, 1],
                                   [63, 65], [64], [100, 1, 1, 27],
                                   [17, 2, 2, 130]])
def test_any_cut_gives_the_same_logits(model, sizes):
    cfg, w, t, want = model
    m = engine(cfg, w)
    assert worst(run(m, t, cut(300, sizes)), want) < EXACT


def test_scratch_smaller_than_the_step(model):
    """A step beyond the scratch rows runs as several batches."""
    cfg, w, t, want = model
    m = engine(cfg, w, prefill_chunk=64)
    assert m.PC == 64
    assert worst(run(m, t), want) < EXACT
    a, b = m.open_sequence(), m.open_sequence()
    got = m.step([entry(a, t[:50]), entry(b, t[:70])]).cpu().numpy()
    assert worst(got, np.concatenate([want[:50], want[:70]])) < EXACT


def test_bf16_whole_model(model):
    cfg, w, t, want = model
    m = engine(cfg, w, "bf16")
    for sizes in ([300], [1], [2, 70, 1]):
        assert rel(run(m, t, cut(300, sizes)), want) < ROUNDED


def test_long_prompt_with_split_keys():
    """Later portions of a long prompt: key splits of runs and tokens."""
    cfg = config([(attention(8, 1, 24, 40), None), (lightning(2), None)])
    w, t = weights(cfg), tokens(cfg, 1500)
    want, _ = Oracle(cfg, w).run(t)
    m = engine(cfg, w, max_seq=1536)
    for cuts in ([1500], [1200, 2, 3, 1, 1, 293], [700, 33, 767]):
        assert worst(run(m, t, cuts), want) < EXACT, cuts
    b = engine(cfg, w, "bf16", max_seq=1536)
    assert rel(run(b, t, [1200, 2, 3, 1, 1, 293]), want) < ROUNDED


def test_mixed_batches_with_reuse(model):
    """Random schedules over four live requests in a pool that is smaller
    than their sum: every logit equals the request's own run."""
    cfg, w, _, _ = model
    o = Oracle(cfg, w)
    reqs = [tokens(cfg, n, 10 + i) for i, n in enumerate(
        [150, 3, 64, 97, 1, 130, 65, 40, 128, 2, 77])]
    want = [o.run(t)[0] for t in reqs]
    m = engine(cfg, w, max_seq=192, pool_tokens=64 * 8)
    rng = np.random.default_rng(5)
    todo, live, at, used = list(range(len(reqs))), {}, {}, set()
    while todo or live:
        while todo and len(live) < 4:
            r = todo[0]
            held = sum(-(-len(reqs[k]) // 64) for k in live)
            if held + -(-len(reqs[r]) // 64) > 8:
                break
            live[todo.pop(0)] = m.open_sequence()
            at[r] = 0
        step, refs = [], []
        for r in rng.permutation(list(live)):
            if len(live) > 1 and rng.random() < 0.2:
                continue                       # left out of this step
            left = len(reqs[r]) - at[r]
            n = min(left, int(rng.choice([1, 1, 2, 3, 17, 63, 64, 65])))
            step.append(entry(live[r], reqs[r][at[r]:at[r] + n]))
            refs.append(want[r][at[r]:at[r] + n])
            at[r] += n
        if not step:
            continue
        got = m.step(step).cpu().numpy()
        assert worst(got, np.concatenate(refs)) < EXACT
        for r in list(live):
            used |= {(r, p) for p in live[r].pages}
            if at[r] == len(reqs[r]):
                m.close_sequence(live.pop(r))
    pages = [p for _, p in used]
    assert len(pages) > len(set(pages))        # pages did change hands
    assert m.cache.free_pages == 8 and m.cache.free_slots == 4


@pytest.mark.parametrize("rows", [2, 3, 5, 9, 16, 19, 40])
def test_many_single_tokens_in_one_step(model, rows):
    """Decode batches of every size class, at unequal lengths."""
    cfg, w, t, want = model
    m = engine(cfg, w, max_batch=rows)
    seqs = [m.open_sequence() for _ in range(rows)]
    lens = [1 + (7 * i) % 90 for i in range(rows)]
    m.step([entry(s, t[:n], []) for s, n in zip(seqs, lens)])
    for k in range(3):
        got = m.step([entry(s, t[n + k:n + k + 1])
                      for s, n in zip(seqs, lens)]).cpu().numpy()
        assert worst(got, np.stack([want[n + k] for n in lens])) < EXACT


def test_wanted_places_and_order(model):
    cfg, w, t, want = model
    m = engine(cfg, w)
    a, b, c = (m.open_sequence() for _ in range(3))
    got = m.step([entry(a, t[:20], [19, 0, 7]), entry(b, t[:1], [0]),
                  entry(c, t[:33], [])]).cpu().numpy()
    assert worst(got, want[[19, 0, 7, 0]]) < EXACT
    assert m.step([entry(c, t[33:40], [])]).shape == (0, cfg["vocab"])
    # one wanted row out of several: the pending additions of that row
    got = m.step([entry(b, t[1:3], [1]), entry(c, t[40:42], [])])
    assert worst(got.cpu().numpy(), want[2:3]) < EXACT


# ----------------------------------------- keys and inputs that stand out

def _needle(at, total, heads=4, kv_heads=2):
    """A model and prompt in which the last token attends to one position
    almost alone: only token 1, placed there, has the key that only token
    2, placed last, asks for."""
    cfg = config([(attention(heads, kv_heads, 24, 40, 0.4, 0.2, 50), None)],
                 width=64)
    w = weights(cfg, 9)
    w["embed"][:, :8] = 0
    w["embed"][2, :4] = w["embed"][1, 4:8] = 3.0
    w["l0.mix.q"][:, 4:8] = w["l0.mix.k"][:, :4] = 0
    w["l0.mix.q.b"][:] = w["l0.mix.k.b"][:] = 0
    d = np.random.default_rng(2).standard_normal(24)
    w["l0.mix.q"][:, :4] = np.tile(d, heads)[:, None] * 2
    w["l0.mix.k"][:, 4:8] = np.tile(d, kv_heads)[:, None] * 2
    w["l0.mix.q.norm"][:] = w["l0.mix.k.norm"][:] = 1.5
    t = 3 + tokens(cfg, total) % (cfg["vocab"] - 3)
    t[at], t[-1] = 1, 2
    return cfg, w, t.astype(np.int32)


@pytest.mark.parametrize("total", [64, 65, 130, 257])
@pytest.mark.parametrize("at", [0, 1, 15, 16, 31, 32, 62, 63, 64, 127, 128])
def test_key_that_stands_out(at, total):
    if at >= total - 1:
        pytest.skip("beyond the prompt")
    cfg, w, t = _needle(at, total)
    o = Oracle(cfg, w)
    want, _ = o.run(t)
    gone = t.copy()
    gone[at] = 3
    assert worst(o.run(gone)[0][-1:], want[-1:]) > 0.1     # it does show
    m = engine(cfg, w)
    for cuts in ([total], [total - 1, 1], [total - 2, 2],
                 cut(total - 1, [50, 3]) + [1]):
        assert worst(run(m, t, cuts)[-1:], want[-1:]) < EXACT
    b = engine(cfg, w, "bf16")
    for cuts in ([total], [total - 1, 1]):
        assert rel(run(b, t, cuts)[-1:], want[-1:]) < ROUNDED


def test_far_key_while_decoding():
    """The asking token comes at every place after a long decode."""
    cfg, w, t = _needle(5, 200, 6, 2)
    o = Oracle(cfg, w)
    m = engine(cfg, w)
    s = m.open_sequence()
    m.step([entry(s, t[:10], [])])
    _, st = o.run(t[:10])
    for k in range(10, 150):
        ask = 2 if k % 9 == 0 else int(t[k])
        z, st = o.run([ask], st)
        got = m.step([entry(s, [ask])]).cpu().numpy()
        assert worst(got, z) < EXACT, k


@pytest.mark.parametrize("every", [1, 3, 32])
def test_query_temperature_edges(every):
    """A large coefficient: a position that takes its neighbour's factor
    differs from the oracle by far more than the tolerance."""
    cfg = config([(attention(4, 2, 24, 40, 0.15, 2.0, every), None)])
    w, t = weights(cfg, 4), tokens(cfg, 100)
    want, _ = Oracle(cfg, w).run(t)
    late = json.loads(json.dumps(cfg))
    late["layers"][0]["mixer"]["q_temp"]["every"] = every + 1
    off, _ = Oracle(late, w).run(t)
    m = engine(cfg, w)
    for cuts in ([100], [1] * 100, cut(100, [2, 31])):
        got = run(m, t, cuts)
        assert worst(got, want) < EXACT
    edge = max(every - 1, 1)
    assert worst(off[edge:], want[edge:]) > 20 * EXACT


@pytest.mark.parametrize("taps", [1, 2, 4, 6])
def test_convolution_window(taps):
    """With closed memory only the convolution looks back: the oldest tap
    is as large as the rest, so an input one place off or lost at a cut
    shows in the row that should see it last, and not in the next."""
    cfg = config([(rglru(40, 2, taps), None)])
    w, t = weights(cfg, 3), tokens(cfg, 80)
    w["l0.mix.lam"][:] = w["l0.mix.ra.b"][:] = 9.0
    w["l0.mix.ra"] *= 0
    w["l0.mix.conv"][:, 0] = 2.0
    o = Oracle(cfg, w)
    want, _ = o.run(t)
    p = 40
    other = t.copy()
    other[p] = (t[p] + 7) % cfg["vocab"]
    diff = np.abs(o.run(other)[0] - want).max(-1)
    assert diff[p + taps - 1] > 0.05 and diff[p + taps:].max() < 1e-6
    m = engine(cfg, w)
    for k in range(p, p + taps + 1):           # a cut at every place
        for cuts in ([k, 80 - k], [k] + [1] * (80 - k), [k, 2, 78 - k]):
            assert worst(run(m, t, cuts), want) < EXACT
            assert worst(run(m, other, cuts), o.run(other)[0]) < EXACT


@pytest.mark.parametrize("kind", ["rglru", "lightning"])
def test_memory_reaches_back(kind):
    """With slow decay the first token still shapes the state 200 tokens
    on; swapping it must show, and the engine must follow."""
    cfg = config([(rglru(48, 3, 2) if kind == "rglru" else
                   lightning(2, 24, 40, [1.0, 0.9999]), None)])
    w, t = weights(cfg), tokens(cfg, 200)
    if kind == "rglru":
        w["l0.mix.lam"][:] = -9.0
    other = t.copy()
    other[0] = (t[0] + 5) % cfg["vocab"]
    o = Oracle(cfg, w)
    want, _ = o.run(t)
    assert worst(o.run(other)[0][-1:], want[-1:]) > 10 * EXACT
    m = engine(cfg, w)
    for cuts in ([200], [199, 1], cut(200, [64, 1, 2])):
        assert worst(run(m, t, cuts), want) < EXACT


def test_first_tokens_after_reuse(model):
    """A slot and pages that a long request left behind: one, two and three
    tokens alone, and the first tokens of a prompt, see none of it."""
    cfg, w, t, want = model
    m = engine(cfg, w, max_batch=1, max_seq=320, pool_tokens=320)
    for cuts in ([1], [2], [3], [1, 1, 1], [1, 2], [2, 1], [90]):
        run(m, t[100:300])
        n = sum(cuts)
        assert worst(run(m, t[:n], cuts), want[:n]) < EXACT


# ---------------------------------------------------- generation and serving

def test_long_greedy_decode_graph_and_eager(model):
    cfg, w, t, _ = model
    want, margin = greedy(cfg, w, t[:5], 180)
    assert margin > 1e-4
    m = engine(cfg, w)
    for graph in (True, False, True):
        m.prefill(t[:5])
        ids = m.decode(180, greedy=True, use_graph=graph)
        assert ids.tolist() == want
    assert m._graph_mode is not None and not getattr(m, "_graph_failed", 0)
    # chunks of the loop, and a token fed by hand afterwards
    m.prefill(t[:5])
    ids = np.concatenate([m.decode(n, greedy=True, first_from_logits=k == 0)
                          for k, n in enumerate([3, 16, 1, 60])])
    assert ids.tolist() == want[:80]


@pytest.mark.parametrize("B", [2, 4, 11])
def test_batched_generation(model, B):
    cfg, w, t, _ = model
    prompts = [t[i:i + 1 + 13 * i % 70] for i in range(B)]
    m = engine(cfg, w, max_batch=B)
    out = m.generate_tokens_batch(prompts, 40)
    for p, ids in zip(prompts, out):
        want, margin = greedy(cfg, w, p, 40)
        assert margin < 1e-4 or ids.tolist() == want


def test_rows_join_and_leave(model):
    """The server's row primitives: join, decode, retire, compact."""
    cfg, w, t, _ = model
    m = engine(cfg, w, max_batch=3)
    prompts = {0: t[:9], 1: t[20:85], 2: t[40:43], 3: t[:70]}
    want = {k: greedy(cfg, w, p, 20)[0] for k, p in prompts.items()}
    got = {}
    for k in (0, 1, 2):
        m.prefill_row(k, prompts[k])
        got[k] = [int(m.bt_next[k].item())]
    for k, ids in zip((0, 1, 2), m.decode_rows(3, 4)):
        got[k] += ids.tolist()
    m.compact_row(0, 2)                        # request 0 leaves
    assert m.rows[2] is None
    for k, ids in zip((2, 1), m.decode_rows(2, 5)):
        got[k] += ids.tolist()
    m.prefill_row(2, prompts[3])
    got[3] = [int(m.bt_next[2].item())]
    for k, ids in zip((2, 1, 3), m.decode_rows(3, 6)):
        got[k] += ids.tolist()
    for k in got:
        assert got[k] == want[k][:len(got[k])], k


def test_generate_session_and_rewind(tmp_path):
    import llm_np_cp_amd as L

    cfg = default(vocab=300)
    w = weights(cfg)
    save(cfg, w, tmp_path / "m")
    tok, m, c = L.load_model(str(tmp_path / "m"), dtype="fp32", max_seq=256)
    p = L.SamplingParams(strategy="greedy")
    prompt = "Once upon a time"
    ids = list(prompt.encode())
    want, _ = greedy(cfg, w, ids, 30)
    fast = L.generate(prompt, tok, m, max_tokens=30, params=p, stream=False)
    slow = L.generate(prompt, tok, m, max_tokens=30, params=p, stream=False,
                      logprobs=2)
    assert fast.token_ids == want and slow.token_ids == want
    assert len(L.generate(prompt, tok, m, max_tokens=12, params=L.
               SamplingParams(strategy="min_p", seed=1), stream=False,
               ).token_ids) == 12
    s = L.ChatSession(tok, m)
    a = s.send("Hi", max_tokens=6).token_ids
    b = s.send("more", max_tokens=6).token_ids
    hist = list(b"Hi")
    assert a == greedy(cfg, w, hist, 6)[0]
    assert b == greedy(cfg, w, hist + a + list(b"more"), 6)[0]
    m.prefill(np.asarray(ids))
    m.rewind(len(ids))
    with pytest.raises(ValueError, match="recurrent"):
        m.rewind(3)


def test_rewind_without_recurrence():
    cfg = config([(attention(), 40), (attention(2, 2), None)], loop=(0, 1, 2))
    w, t = weights(cfg), tokens(cfg, 40)
    m = engine(cfg, w)
    m.prefill(t)
    m.rewind(25)
    want, _ = Oracle(cfg, w).run(np.concatenate([t[:25], t[:9]]))
    assert worst(m.forward_positions(t[:9], 25), want[25:]) < EXACT


def test_server_batches_requests(tmp_path):
    """The HTTP scheduler: concurrent greedy requests in one lockstep
    group give what each gives alone."""
    pytest.importorskip("fastapi")
    from concurrent.futures import ThreadPoolExecutor

    from fastapi.testclient import TestClient

    from llm_np_cp_amd.runtime.server import build_app

    cfg = config([(attention(), 60), (rglru(), None), (lightning(), 72)],
                 vocab=280)
    w = weights(cfg)
    save(cfg, w, tmp_path / "m")
    app = build_app(str(tmp_path / "m"), backend="gpu", dtype="fp32",
                    max_seq=256, max_batch=3, batch_window_ms=60)
    prompts = ["a", "hello there", "x" * 70, "four", "The end."]
    want = [bytes(i % 256 for i in greedy(cfg, w, list(p.encode()), 12)[0])
            .decode("utf-8", errors="replace") for p in prompts]
    with TestClient(app) as c:
        def ask(p):
            return c.post("/v1/completions", json={
                "prompt": p, "max_tokens": 12, "strategy": "greedy",
                "stop_on_eos": False}).json()["choices"][0]["text"]
        with ThreadPoolExecutor(5) as ex:
            got = list(ex.map(ask, prompts))
        assert got == want
        assert c.get("/stats").json()["max_group"] > 1


def test_command_line(tmp_path):
    cfg = config([(attention(), 60), (rglru(), None)], vocab=300)
    w = weights(cfg)
    save(cfg, w, tmp_path / "m")
    p = subprocess.run(
        [sys.executable, "-m", "llm_np_cp_amd", "abc", "--model",
         str(tmp_path / "m"), "--backend", "gpu", "--dtype", "fp32",
         "--strategy", "greedy", "--max-tokens", "8"], cwd=ROOT,
        capture_output=True, timeout=100)
    assert p.returncode == 0, p.stderr.decode()[-2000:]
    want, _ = greedy(cfg, w, list(b"abc"), 8)
    text = bytes(i % 256 for i in want).decode("utf-8", errors="replace")
    assert text in p.stdout.decode("utf-8", errors="replace")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_trace_run(tmp_path, dtype):
    """The command: portions beside single tokens, slots given back and
    taken again, more requests over time than slots."""
    cfg = default()
    w = weights(cfg)
    save(cfg, w, tmp_path / "m")
    (tmp_path / "out").mkdir()
    o = Oracle(cfg, w)
    reqs = {f"q{i}": tokens(cfg, n, i) for i, n in enumerate(
        [70, 5, 64, 2, 66, 30])}
    plan = [{"q0": 66, "q1": 2, "q2": 1}, {"q0": 1, "q1": 2, "q2": 60},
            {"q0": 1, "q3": 2, "q1": 1}, {"q2": 3, "q4": 65}, {"q0": 2},
            {"q4": 1, "q5": 29}, {"q5": 1}]
    at, lines, refs = dict.fromkeys(reqs, 0), [], []
    full = {k: o.run(t)[0] for k, t in reqs.items()}
    for n, step in enumerate(plan):
        entries, end, rows = [], [], []
        for k, c in step.items():
            lo, hi = at[k], at[k] + c
            want = [] if n == 3 else [c - 1] if c < 4 else [0, c - 1]
            entries.append({"id": k, "tokens": reqs[k][lo:hi].tolist(),
                            "want": want})
            rows += [full[k][lo + x] for x in want]
            at[k] = hi
            if hi == len(reqs[k]):
                end.append(k)
        lines.append(json.dumps({"step": n, "entries": entries, "end": end}))
        refs.append(rows)
    assert all(at[k] == len(reqs[k]) for k in reqs)
    p = subprocess.run(
        [os.path.join(ROOT, "bin", "trace_run"), "--model",
         str(tmp_path / "m"), "--dtype", dtype, "--out",
         str(tmp_path / "out"), "--max-tokens", "320"],
        input=("\n".join(lines) + "\n").encode(), capture_output=True,
        timeout=100)
    assert p.returncode == 0, p.stderr.decode()[-2000:]
    done = [l for l in p.stdout.decode().splitlines() if l.startswith("done")]
    assert done == [f"done {n}" for n in range(len(plan))]
    for n, rows in enumerate(refs):
        f = tmp_path / "out" / f"{n}.f32"
        assert f.exists() == bool(rows)
        if rows:
            got = np.fromfile(f, "<f4").reshape(-1, cfg["vocab"])
            if dtype == "float32":
                assert worst(got, np.stack(rows)) < EXACT
            else:
                assert rel(got, np.stack(rows)) < ROUNDED
