"""What the performance of this framework is measured on.

A case is one thing a program does with a loaded model: read a prompt,
answer it, answer several at once, or check the tokens that a draft model
proposed.  The models are the architectures of the presets with their own
widths, heads, windows and soft caps; all but the flagship have fewer
layers and a vocabulary of 32768, so that one fits beside two others and
is made in a second (every layer of a model is alike, so a pass is a
stretch of the full model's).

Weights are random with the statistics of a trained checkpoint: normed
projections of unit scale, a residual stream that every layer changes by a
fraction, and a head that is sure of its next token, so a rounding never
changes the text and logits after it can be compared.
"""

import dataclasses
import math
import zlib

import numpy as np
import torch

import llm_np_cp_amd as L
from llm_np_cp_amd.io.loader import hf_weight_shapes
from llm_np_cp_amd.models.registry import engine_class

VOCAB = 32768

# name -> (preset, what differs from it)
MODELS = {
    "llama-1b": ("llama-3.2-1b", {}),
    "llama-3b": ("llama-3.2-3b", dict(num_hidden_layers=3, vocab_size=VOCAB)),
    "llama-8b": ("llama-3.1-8b", dict(num_hidden_layers=2, vocab_size=VOCAB)),
    "gemma-2b": ("gemma-2-2b", dict(num_hidden_layers=4, vocab_size=VOCAB)),
    "gemma-9b": ("gemma-2-9b", dict(num_hidden_layers=2, vocab_size=VOCAB)),
    "qwen-7b": ("qwen2.5-7b", dict(num_hidden_layers=2, vocab_size=VOCAB)),
    "mistral-7b": ("mistral-7b", dict(num_hidden_layers=2)),
    # eight experts, two a token, at half the width
    "mixtral": ("mixtral-8x7b", dict(
        num_hidden_layers=2, hidden_size=2048, intermediate_size=4096,
        num_attention_heads=16, num_key_value_heads=4)),
    # grouped attention, gated and decaying linear recurrences
    "garupel-2k": ("garupel-2k", {}),
}

LISTED = [
    # the smallest calls: one check of four proposed tokens and the last
    # one, as speculative decoding makes after every four draft steps
    dict(name="verify 3b bf16", do="verify", model="llama-3b", dtype="bf16",
         kv="bf16", prompt=901, new=5, batch=1),
    # time to the first token of a chat message on the flagship
    dict(name="message 1b bf16", do="prompt", model="llama-1b",
         dtype="bf16", kv="bf16", prompt=37, new=0, batch=1),
    # a chat turn on the flagship, token by token
    dict(name="turn 1b bf16", do="answer", model="llama-1b", dtype="bf16",
         kv="bf16", prompt=61, new=48, batch=1),
    # a page of text read by the flagship
    dict(name="page 1b bf16", do="prompt", model="llama-1b", dtype="bf16",
         kv="bf16", prompt=1999, new=0, batch=1),
    # a long document read at 8B width
    dict(name="document 8b bf16", do="prompt", model="llama-8b",
         dtype="bf16", kv="bf16", prompt=8187, new=0, batch=1),
    # a document longer than the sliding window, soft-capped scores
    dict(name="window 2b bf16", do="prompt", model="gemma-2b", dtype="bf16",
         kv="bf16", prompt=5003, new=0, batch=1),
    # a question about a document: quantised weights and cache
    dict(name="question 8b fp8", do="answer", model="llama-8b", dtype="fp8",
         kv="fp8", prompt=6001, new=64, batch=1),
    # the smallest weights, one sequence
    dict(name="turn 7b fp4", do="answer", model="mistral-7b", dtype="fp4",
         kv="bf16", prompt=130, new=48, batch=1),
    # a full serving group of quantised rows
    dict(name="group 9b fp8", do="answer", model="gemma-9b", dtype="fp8",
         kv="bf16", prompt=611, new=32, batch=16),
    # a serving group without quantisation, biased projections
    dict(name="group 7b bf16", do="answer", model="qwen-7b", dtype="bf16",
         kv="bf16", prompt=333, new=24, batch=6),
    # routed experts: a prompt, then token by token
    dict(name="experts bf16", do="answer", model="mixtral", dtype="bf16",
         kv="bf16", prompt=1100, new=24, batch=1),
    # a group of the layer-list designs: ragged prompts in one batch
    dict(name="layers 2k bf16", do="answer", model="garupel-2k",
         dtype="bf16", kv="bf16", prompt=501, new=24, batch=4),
]

# model -> (weights, caches, longest prompt, largest group); a longest
# prompt keeps a drawn case below the largest listed one
RANGES = {
    "llama-1b": (("bf16", "fp8"), ("bf16",), 2048, 1),
    "llama-3b": (("bf16", "fp8", "fp4"), ("bf16",), 4096, 4),
    "llama-8b": (("bf16", "fp8"), ("bf16", "fp8"), 6144, 12),
    "gemma-2b": (("bf16", "fp8"), ("bf16", "fp8"), 5120, 4),
    "gemma-9b": (("bf16", "fp8"), ("bf16",), 2048, 16),
    "qwen-7b": (("bf16", "fp8"), ("bf16",), 2048, 8),
    "mistral-7b": (("bf16", "fp8", "fp4"), ("bf16", "fp8"), 5120, 8),
    "mixtral": (("bf16", "fp8"), ("bf16",), 1400, 4),
    "garupel-2k": (("bf16",), ("bf16",), 700, 4),
}


def listed():
    return [dict(c) for c in LISTED]


def _spread(rng, lo, hi):
    """A whole number, evenly over the logarithm."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo),
                                            math.log(hi + 1)))))


def draw(rng):
    model = rng.choice(sorted(RANGES))
    weights, caches, longest, group = RANGES[model]
    c = dict(do=rng.choice(("prompt", "answer", "answer", "verify")),
             model=model, dtype=rng.choice(weights), kv=rng.choice(caches),
             prompt=_spread(rng, 2, longest), new=0, batch=1)
    if model == "garupel-2k":      # a recurrence cannot be rolled back
        c["do"] = rng.choice(("prompt", "answer"))
    if c["do"] == "verify":
        c["new"] = rng.randint(2, 9)
    if c["do"] == "answer":
        c["new"] = _spread(rng, 3, 48)
        # a group is read row by row; the rows share the longest prompt
        if c["dtype"] != "fp4" and rng.random() < 0.5:
            c["batch"] = rng.randint(1, group)
            c["prompt"] = max(2, min(c["prompt"], longest // c["batch"]))
    return c


# ----------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------

def _config(case):
    preset, other = MODELS[case["model"]]
    cfg = L.preset_config(preset)
    if other:
        cfg = dataclasses.replace(cfg, layer_types=[], **other)
    return cfg


class Checkpoint:
    """Tensors by name, each a stretch of one long cycle of normals (bf16
    values), so that a checkpoint is made at the speed of a copy."""

    CYCLE = 4194301      # prime: no two rows are the same stretch

    def __init__(self, cfg, seed):
        self.cfg, self.shapes = cfg, hf_weight_shapes(cfg)
        self.layered = not hasattr(cfg, "head_dim")
        rng = np.random.default_rng(seed)
        self.cycle = torch.from_numpy(
            rng.standard_normal(self.CYCLE, dtype=np.float32))
        self.seed, self.scaled = seed, {}

    def _values(self, shape, start, scale, base=0.0):
        key = (scale, base)
        if key not in self.scaled:
            self.scaled[key] = (self.cycle * scale + base).bfloat16().half() \
                .numpy()
        pool, n = self.scaled[key], int(np.prod(shape))
        out = np.empty(n, np.float16)
        at, start = 0, start % self.CYCLE
        while at < n:
            m = min(n - at, self.CYCLE - start)
            out[at:at + m] = pool[start:start + m]
            at, start = at + m, 0
        return out.reshape(shape)

    def _spot(self, name):
        return zlib.crc32(f"{name}/{self.seed}".encode())

    def __getitem__(self, name):
        shape, cfg = self.shapes[name], self.cfg
        spot = self._spot(name)
        H = cfg.hidden_size
        if name in ("embed", "head", "model.embed_tokens.weight",
                    "lm_head.weight"):
            # row t of the head is the embedding of t - 1: t - 1 is
            # followed by t (by itself, where the two are one tensor)
            spot = self._spot("embed")
            if "head" in name:
                spot = spot % self.CYCLE + self.CYCLE - H
            if self.layered:
                return self._values(shape, spot,
                                    1.0 if name == "embed" else 0.02)
            return self._values(shape, spot, H ** -0.5 if
                                cfg.model_type == "gemma2" else 0.02)
        if self.layered:
            if name.endswith("lam"):          # slow and fast forgetting
                return self._values(shape, spot, 1.0, -4.0)
            if "norm" in name:
                return self._values(shape, spot, 0.02, 0.2 if
                                    name.endswith(("norm1b", "norm2b"))
                                    else 1.0)
            if name.endswith(".b"):
                return self._values(shape, spot, 0.1)
            return self._values(shape, spot, shape[-1] ** -0.5)
        if "norm" in name:
            base = 1.0
            if cfg.model_type == "gemma2":    # stored without the one
                base = (-0.8 if "post" in name else 0.0)
            return self._values(shape, spot, 0.05, base)
        if name.endswith("bias"):
            return self._values(shape, spot, 0.2)
        scale = shape[-1] ** -0.5
        if "o_proj" in name or "down_proj" in name or ".w2." in name:
            scale *= 0.01 if cfg.model_type != "gemma2" else 1.0
        return self._values(shape, spot, scale)

    def __contains__(self, name):
        return name in self.shapes

    def keys(self):
        return self.shapes.keys()

    def get(self, name, default=None):
        return self[name] if name in self.shapes else default


def _texts(case, seed, vocab):
    """The prompts, rows of a group shorter and shorter down to a half,
    and the tokens to check."""
    rng = np.random.default_rng((seed, 1))
    B, P = case["batch"], case["prompt"]
    texts = [rng.integers(0, vocab, size=max(1, P - b * P // (2 * B)))
             for b in range(B)]
    return texts, rng.integers(0, vocab, size=case["new"])


def prepare(case, seed):
    cfg = _config(case)
    texts, proposed = _texts(case, seed, cfg.vocab_size)
    room = case["prompt"] + case["new"] + 64
    model = engine_class(cfg)(
        cfg, Checkpoint(cfg, seed), dtype=case["dtype"], max_seq=room,
        kv_dtype=case["kv"], max_batch=case["batch"])
    if case["do"] == "verify":
        model.prefill(texts[0])
    return {"case": case, "model": model, "texts": texts,
            "proposed": proposed}


def run(state):
    case, model, texts = state["case"], state["model"], state["texts"]
    if case["do"] == "prompt":
        _, logits = model.prefill(texts[0])
        return {"logits": logits}
    if case["do"] == "verify":
        model.rewind(case["prompt"])
        return {"logits": model.forward_positions(state["proposed"],
                                                  case["prompt"])}
    if case["batch"] == 1:
        ids = model.generate_tokens(texts[0], case["new"], greedy=False,
                                    min_p=0.1)
        return {"ids": np.asarray(ids), "logits": model.b_logits}
    ids = model.generate_tokens_batch(texts, case["new"])
    logits = getattr(model, "bt_logits", None)      # in bf16, where it has it
    if logits is None:
        logits = model.bt_logits32
    return {"ids": ids, "logits": logits[:case["batch"]]}


# ----------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------

WEIGHT_BYTES = {"bf16": 2.0, "fp8": 1.0, "fp4": 0.5 + 1 / 32}


def work(case):
    cfg = _config(case)
    shapes = hf_weight_shapes(cfg)
    head = cfg.vocab_size * cfg.hidden_size
    mats = {n: float(np.prod(s)) for n, s in shapes.items()
            if len(s) >= 2 and "embed" not in n and "head" not in n}
    experts = sum(v for n, v in mats.items() if ".experts." in n)
    rest = sum(mats.values()) - experts
    if hasattr(cfg, "head_dim"):
        E, top = cfg.num_local_experts or 1, cfg.num_experts_per_tok
        spans = [cfg.sliding_window if cfg.is_sliding(i) else 1 << 30
                 for i in range(cfg.num_hidden_layers)]
        per_key = 4 * cfg.num_attention_heads * cfg.head_dim
        kv = (2 * cfg.num_key_value_heads * cfg.head_dim
              * (1 if case["kv"] == "fp8" else 2))
    else:
        E = top = 1
        mix = [l.mixer for l in cfg.layers if l.mixer.kind == "attention"]
        spans = [1 << 30] * len(mix)
        per_key = 2 * mix[0].heads * (mix[0].dim + mix[0].vdim)
        kv = 2 * mix[0].kv_heads * (mix[0].dim + mix[0].vdim)
    wb = WEIGHT_BYTES[case["dtype"]]
    nbytes = flops = 0.0

    def step(rows, logits):
        """One reading of the weights; rows: (first position, tokens)."""
        nonlocal nbytes, flops
        n = sum(k for _, k in rows)
        used = min(E, n * top) / E if E > 1 else 1.0
        nbytes += wb * (rest + experts * used)
        flops += 2.0 * n * (rest + experts * (top / E if E > 1 else 1.0))
        if logits:
            nbytes += wb * head
            flops += 2.0 * logits * head
        for p, k in rows:
            for span in spans:
                # keys that token p + j sees: min(p + j + 1, span)
                ramp = max(0, min(k, span - p))
                keys = ramp * p + ramp * (ramp + 1) / 2 + (k - ramp) * span
                flops += per_key * keys
                nbytes += kv * (min(p, span) + k)

    texts, _ = _texts(case, 0, cfg.vocab_size)
    lens = [len(t) for t in texts]
    if case["do"] == "verify":
        step([(case["prompt"], case["new"])], case["new"])
    else:
        step([(0, n) for n in lens], len(lens))
    for j in range(case["new"] - 1 if case["do"] == "answer" else 0):
        step([(n + j, 1) for n in lens], len(lens))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the logits of one pass were off the 64-bit
    ones, and off those of another pass with its sums in another order:
    0.012 over the sixteen layers of the flagship, 0.006 over the few of
    the other models in bf16 (a token's last expert may change with a
    tie), 0.032 where activations are rounded to fp8.  The largest
    difference was 4.5 times the mean one."""
    rel = 0.02
    if case["model"] in ("llama-1b", "mixtral"):
        rel = 0.05
    if case["dtype"] == "fp8":
        rel = 0.12
    return {"rel": rel, "max": 5 * rel, "differ": 0.0}


# ----------------------------------------------------------------------
# the same in 64 bits
# ----------------------------------------------------------------------

def _as_e4m3(w):
    """Rows scaled to 448."""
    s = w.abs().amax(dim=1, keepdim=True).clamp(min=1e-8).float() / 448.0
    q = (w.float() * (1.0 / s)).to(torch.float8_e4m3fn)
    return q.double() * s.double()


def _as_mxfp4(w):
    """Blocks of 32 with the least power of two that holds them."""
    b = w.double().reshape(-1, 32)
    top = b.abs().amax(dim=1, keepdim=True)
    e = torch.ceil(torch.log2(top.clamp(min=2.0 ** -126) / 6.0))
    s = torch.exp2(e.clamp(-126, 127))
    grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0],
                        dtype=torch.float64, device=w.device)
    mid = (grid[1:] + grid[:-1]) / 2
    a = (b / s).abs()
    code = torch.searchsorted(mid, a)                  # halves stay below
    tie = (code < 7) & (a == mid[code.clamp(max=6)]) & (code % 2 == 1)
    return (grid[(code + tie).clamp(max=7)] * s * b.sign()).reshape(w.shape)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, p, span=1 << 30, cap=0.0):
    """q [T, heads, d] at positions p, ..; k, v [keys, kv heads, d]."""
    T, n, g = q.shape[0], q.shape[1], q.shape[1] // k.shape[1]
    kh = k.permute(1, 2, 0).repeat_interleave(g, 0).contiguous()
    vh = v.permute(1, 0, 2).repeat_interleave(g, 0).contiguous()
    out = torch.empty(T, n, v.shape[2], dtype=q.dtype, device=q.device)
    j = torch.arange(k.shape[0], device=q.device)
    for a in range(0, T, 512):
        z = q[a:a + 512].permute(1, 0, 2).contiguous()
        s = torch.matmul(z, kh) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        i = (p + a + torch.arange(z.shape[1], device=q.device))[:, None]
        s = s.masked_fill((j > i) | (j <= i - span), -math.inf)
        out[a:a + 512] = torch.matmul(torch.softmax(s, -1), vh) \
            .permute(1, 0, 2)
    return out.reshape(T, -1)


class Transformer:
    """The dense and routed transformers; state: keys and values."""

    def __init__(self, cfg, ckpt, dtype):
        self.cfg, gemma = cfg, cfg.model_type == "gemma2"
        self.w = {}
        for n in ckpt.keys():
            t = torch.from_numpy(ckpt[n]).cuda()
            if "norm" in n:
                t = t.double() + (1.0 if gemma else 0.0)
            elif t.dim() == 1 or "embed" in n or "gate.weight" in n:
                t = t.double()        # never quantised
            elif dtype == "fp8":
                t = _as_e4m3(t.bfloat16())
            elif dtype == "fp4":
                t = _as_mxfp4(t)
            else:
                t = t.double()
            self.w[n] = t
        self.head = self.w.get("lm_head.weight")
        if self.head is None:
            self.head = torch.from_numpy(
                ckpt["model.embed_tokens.weight"]).cuda()
            self.head = (_as_e4m3(self.head.bfloat16()) if dtype == "fp8"
                         else _as_mxfp4(self.head) if dtype == "fp4"
                         else self.head.double())
        self.freq = torch.from_numpy(np.asarray(self._frequencies())).cuda()

    def _frequencies(self):
        c = self.cfg
        f = c.rope_theta ** (-np.arange(0, c.head_dim, 2) / c.head_dim)
        r = c.rope_scaling
        if not r:
            return f
        # long waves are stretched, short ones stay, a ramp between
        turns = r["original_max_position_embeddings"] * f / (2 * math.pi)
        ramp = np.clip((turns - r["low_freq_factor"]) /
                       (r["high_freq_factor"] - r["low_freq_factor"]), 0, 1)
        return f * ((1 - ramp) / r["factor"] + ramp)

    def _rotate(self, x, p):
        a = (p + torch.arange(len(x), device=x.device))[:, None] * self.freq
        c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
        u, v = x.chunk(2, -1)
        return torch.cat([u * c - v * s, v * c + u * s], -1)

    def _mlp(self, p, x):
        c, w = self.cfg, self.w
        act = (torch.nn.functional.silu if c.hidden_act == "silu" else
               lambda z: torch.nn.functional.gelu(z, approximate="tanh"))
        if not c.is_moe:
            m = p + "mlp."
            return (act(x @ w[m + "gate_proj.weight"].T) *
                    (x @ w[m + "up_proj.weight"].T)) @ \
                w[m + "down_proj.weight"].T
        m = p + "block_sparse_moe."
        z = x @ w[m + "gate.weight"].T
        val, idx = z.topk(c.num_experts_per_tok, -1)
        share = torch.softmax(val, -1)
        y = torch.zeros_like(x)
        for e in range(c.num_local_experts):
            row, which = (idx == e).nonzero(as_tuple=True)
            q = f"{m}experts.{e}."
            h = (act(x[row] @ w[q + "w1.weight"].T) *
                 (x[row] @ w[q + "w3.weight"].T)) @ w[q + "w2.weight"].T
            y.index_add_(0, row, h * share[row, which][:, None])
        return y

    def run(self, ids, state, last=True):
        c, w = self.cfg, self.w
        gemma, eps, hd = c.model_type == "gemma2", c.rms_norm_eps, c.head_dim
        p0 = 0 if state is None else len(state[0][0])
        x = w["model.embed_tokens.weight"][
            torch.as_tensor(np.asarray(ids), device="cuda").long()]
        x = x * (math.sqrt(c.hidden_size) if gemma else 1.0)
        new = []
        for i in range(c.num_hidden_layers):
            p = f"model.layers.{i}."
            a = p + "self_attn."
            norm = lambda z, n: _rms(z, eps) * w[p + n + ".weight"]
            h = norm(x, "input_layernorm")
            q, k, v = (h @ w[f"{a}{n}_proj.weight"].T +
                       w.get(f"{a}{n}_proj.bias", 0.0) for n in "qkv")
            q, k, v = (t.reshape(len(x), -1, hd) for t in (q, k, v))
            q, k = self._rotate(q, p0), self._rotate(k, p0)
            if state is not None:
                k = torch.cat([state[i][0], k])
                v = torch.cat([state[i][1], v])
            new.append((k, v))
            scale = hd ** -0.5
            if gemma:
                scale = c.query_pre_attn_scalar ** -0.5
            o = _attend(q, k, v, scale, p0,
                        c.sliding_window if c.is_sliding(i) else 1 << 30,
                        c.attn_logit_softcapping or 0.0)
            o = o @ w[a + "o_proj.weight"].T
            if gemma:
                x = x + norm(o, "post_attention_layernorm")
                y = self._mlp(p, norm(x, "pre_feedforward_layernorm"))
                x = x + norm(y, "post_feedforward_layernorm")
            else:
                x = x + o
                x = x + self._mlp(p, norm(x, "post_attention_layernorm"))
        x = x[-1:] if last else x
        z = (_rms(x, eps) * w["model.norm.weight"]) @ self.head.T
        cap = c.final_logit_softcapping
        return (cap * torch.tanh(z / cap) if cap else z), new


class Recurrent:
    """Garupel: sandwich-normed layers of attention with normed queries
    and keys, a gated recurrence behind a convolution, or linear attention
    with a decay per head; state: one entry a layer."""

    def __init__(self, cfg, ckpt, dtype):
        self.cfg = cfg
        self.w = {n: torch.from_numpy(ckpt[n]).cuda().double()
                  for n in ckpt.keys()}

    def _attention(self, p, m, h, st):
        w, eps, T = self.w, self.cfg.norm_eps, len(h)
        p0 = 0 if st is None else len(st[0])
        q, k, v = (h @ w[p + n].T + w[p + n + ".b"] for n in "qkv")
        q = _rms(q, eps) * w[p + "q.norm"]
        k = _rms(k, eps) * w[p + "k.norm"]
        pos = p0 + torch.arange(T, device=h.device)
        qt = m.to_dict()["q_temp"]
        t = 1.0 + qt["coef"] * torch.log(
            torch.floor((pos + 1) / qt["every"]) + 1.0).double()
        q = (q * t[:, None]).reshape(T, m.heads, m.dim)
        k = k.reshape(T, m.kv_heads, m.dim)
        v = v.reshape(T, m.kv_heads, m.vdim)
        if st is not None:
            k, v = torch.cat([st[0], k]), torch.cat([st[1], v])
        o = _attend(q, k, v, m.scale, p0)
        return (o * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T, (k, v)

    def _rglru(self, p, m, h, st):
        w, T = self.w, len(h)
        n, nb, taps = m.width, m.blocks, w[p + "conv"].shape[1]
        if st is None:
            st = h.new_zeros(n), h.new_zeros(taps - 1, n)
        y = torch.nn.functional.gelu(h @ w[p + "y"].T + w[p + "y.b"],
                                     approximate="tanh")
        full = torch.cat([st[1], h @ w[p + "x"].T + w[p + "x.b"]])
        u = w[p + "conv.b"] + sum(full[j:j + T] * w[p + "conv"][:, j]
                                  for j in range(taps))
        ub = u.reshape(T, nb, n // nb).permute(1, 2, 0).contiguous()
        r, i = (torch.sigmoid(
            torch.matmul(w[p + g], ub) + w[p + g + ".b"][:, :, None])
            .permute(2, 0, 1).reshape(T, n) for g in ("ra", "ri"))
        log_a = -8.0 * r * torch.nn.functional.softplus(w[p + "lam"])
        a = torch.exp(log_a)
        add = torch.sqrt(-torch.expm1(2.0 * log_a)) * i * u
        s, out = st[0], []
        for t in range(T):
            s = torch.addcmul(add[t], a[t], s)
            out.append(s)
        return ((torch.stack(out) * y) @ w[p + "o"].T,
                (s, full[T:]))

    def _lightning(self, p, m, h, st):
        w, T = self.w, len(h)
        q, k, v = (torch.nn.functional.silu(h @ w[p + n].T)
                   .reshape(T, m.heads, -1) for n in "qkv")
        decay = torch.tensor(m.to_dict()["decay"], dtype=h.dtype,
                             device=h.device)
        # o_t = sum over j <= t of decay^(t - j) (q_t . k_j) v_j, and what
        # the state brings
        t = torch.arange(T, device=h.device, dtype=h.dtype)
        gap = t[:, None] - t[None]
        mask = torch.where(gap >= 0, decay[:, None, None] **
                           gap.clamp(min=0), torch.zeros_like(gap))
        qh, kh, vh = (z.permute(1, 0, 2).contiguous() for z in (q, k, v))
        o = torch.matmul(
            torch.matmul(qh, kh.transpose(1, 2).contiguous()) * mask, vh)
        left = decay[:, None] ** (T - 1 - t)             # [heads, T]
        s = torch.matmul((kh * left[..., None]).transpose(1, 2).contiguous(),
                         vh)
        if st is not None:
            o = o + torch.matmul(qh * (decay[:, None] ** (t + 1))[..., None],
                                 st)
            s = s + st * (decay ** T)[:, None, None]
        o = o.permute(1, 0, 2).reshape(T, -1)
        y = _rms(o, self.cfg.norm_eps) * w[p + "norm"]
        return (y * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T, s

    def run(self, ids, state, last=True):
        c, w = self.cfg, self.w
        norm = lambda z, n: _rms(z, c.norm_eps) * w[n]
        x = w["embed"][torch.as_tensor(np.asarray(ids), device="cuda").long()]
        new = []
        for i, l in enumerate(c.layers):
            p = f"l{i}."
            f = {"attention": self._attention, "rglru": self._rglru,
                 "lightning": self._lightning}[l.mixer.kind]
            y, st = f(p + "mix.", l.mixer, norm(x, p + "norm1"),
                      None if state is None else state[i])
            new.append(st)
            x = x + norm(y, p + "norm1b")
            up = torch.relu(norm(x, p + "norm2") @ w[p + "mlp.up"].T)
            x = x + norm((up * up) @ w[p + "mlp.down"].T, p + "norm2b")
        x = x[-1:] if last else x
        return norm(x, "final.norm") @ w["head"].T, new


def exact(case, seed):
    cfg = _config(case)
    texts, proposed = _texts(case, seed, cfg.vocab_size)
    kind = Transformer if hasattr(cfg, "head_dim") else Recurrent
    model = kind(cfg, Checkpoint(cfg, seed), case["dtype"])
    if case["do"] == "prompt":
        return {"logits": model.run(texts[0], None)[0].cpu().numpy()}
    if case["do"] == "verify":
        _, st = model.run(texts[0], None)
        return {"logits": model.run(proposed, st, last=False)[0]
                .cpu().numpy()}
    ids, logits = [], []
    for t in texts:
        z, st = model.run(t, None)
        out = [int(z.argmax())]
        for _ in range(case["new"] - 1):
            z, st = model.run(out[-1:], st)
            out.append(int(z.argmax()))
        ids.append(out)
        logits.append(z[0])
    if case["batch"] == 1:
        return {"ids": np.asarray(ids[0]), "logits": logits[0]}
    return {"ids": np.asarray(ids), "logits": torch.stack(logits)}
