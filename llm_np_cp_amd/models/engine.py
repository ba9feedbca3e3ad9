"""GPU inference engine: Llama-3.2 / Gemma-2 forward on hand-written
CDNA4 HIP kernels, PyTorch tensors as memory containers only.

MI355X-first design:
  - every compute op is a kernel of this repository (``csrc/``: products
    of one row, of few and of many, attention of prompts and of new
    tokens, norms, router, sampler) — no ATen math in the forward pass, no eager fallback (ops fail loudly if the
    extension is missing);
  - preallocated KV pool per layer (in-place writes, no concat);
  - decode state (seq length, sampled token, RNG counter, output ring)
    lives in device memory so a decode step has zero host round-trips and
    is replayed: its launches, or a hipGraph of them (torch.cuda.CUDAGraph);
  - tensor parallelism: head/row/col-sharded weights per rank, RCCL
    all-reduce after o_proj and down_proj, all-gather for logits
    (world_size==1 skips collectives — same code path).

Reference parity: this replaces the CuPy model classes
(``/root/reference/llama3.2_model.py:334-822``) — same capability
(forward with KV cache, returns logits), built from the architectural
spec of the two families rather than translated.
"""

from __future__ import annotations

from typing import Dict, Optional

import numpy as np
import torch

from ..core.config import ModelConfig
from ..ops import hip_ops as ho
from ..parallel import tp as tpu
from .decode_loop import DecodeLoop, DeviceCacheHandle


class GPUModel(DecodeLoop):
    def __init__(self, config: ModelConfig, weights: Dict[str, np.ndarray],
                 dtype: str = "bf16", max_seq: Optional[int] = 4096,
                 prefill_chunk: int = 2048, device: Optional[str] = None,
                 seed: int = 0, force_tp_path: bool = False,
                 kv_dtype: str = "bf16", max_batch: int = 1):
        """``max_seq=None`` sizes the KV pool from FREE HBM after the
        weights land (288 GB per MI355X), capped
        at config.max_position_embeddings.  ``max_batch>1`` allocates
        per-sequence KV pools for lockstep batched decode
        (prefill_batch/decode_batch; beyond-parity serving capability)."""
        if not torch.cuda.is_available():
            raise RuntimeError("GPUModel requires a GPU (MI355X)")
        self.config = config
        self.seed = seed
        assert 1 <= max_batch <= 256
        self.max_batch = max_batch
        self._pb = 0  # current sequence row during per-sequence prefill
        self.dtype = dtype
        if dtype not in ("bf16", "fp8", "fp4"):
            raise ValueError(f"unsupported dtype {dtype!r}")
        # fp4 = MXFP4 weights for decode steps of one sequence (half the
        # fp8 stream) and for prompts; a group's decode steps run on an
        # fp8 copy (the fp8 machinery flag covers both quantized modes)
        self.fp8 = dtype in ("fp8", "fp4")
        self.wq4 = dtype == "fp4"
        # fp4 + batch pools: a group's decode steps run on fp8, so keep
        # the fp8 copy only then; max_batch=1 fp4 engines are SINGLE-COPY
        self.keep_fp8 = (dtype == "fp8") or (self.wq4 and max_batch > 1)
        if kv_dtype not in ("bf16", "fp8"):
            raise ValueError(f"unsupported kv_dtype {kv_dtype!r}")
        self.kv_dtype = kv_dtype
        self.kv8 = kv_dtype == "fp8"  # e4m3 KV pool, per-(head,pos) scales
        # Mixtral sparse MoE: per-token top-k routed experts (one row:
        # products indexed by the device's choice; more: rows sorted by
        # expert, each expert over its own)
        self.moe = config.is_moe
        self.topk = config.num_experts_per_tok
        if self.moe:
            if self.wq4:
                raise ValueError("MoE + fp4 weights not supported yet")
            if config.model_type == "gemma2":
                raise ValueError("MoE is a llama-family (Mixtral) feature")
        self.rank, self.world = tpu.init_distributed()
        # exercise the TP code path on 1 GPU (collectives no-op at
        # world=1, partial sums are then exact) — used by tests
        self.tp_branch = self.world > 1 or force_tp_path
        if device is None:
            device = f"cuda:{self.rank % max(torch.cuda.device_count(), 1)}"
        self.device = torch.device(device)
        torch.cuda.set_device(self.device)

        cfg = config
        tp = self.world
        assert cfg.num_attention_heads % tp == 0, "nh must divide tp"
        assert cfg.num_key_value_heads % tp == 0, \
            f"kv heads {cfg.num_key_value_heads} not divisible by tp {tp}"
        assert cfg.intermediate_size % tp == 0
        assert cfg.vocab_size % tp == 0
        if self.moe and tp > 1:
            raise ValueError("MoE tensor parallelism (expert parallel) "
                             "is not implemented yet — run TP=1")
        self.nh_l = cfg.num_attention_heads // tp
        self.kvh_l = cfg.num_key_value_heads // tp
        self.inter_l = cfg.intermediate_size // tp
        self.vocab_l = cfg.vocab_size // tp
        self.hd = cfg.head_dim
        self.H = cfg.hidden_size

        # one-shot xGMI collectives for decode-sized payloads (validated
        # on hardware at init; silent RCCL fallback when unavailable)
        if self.world > 1:
            slot_bytes = max(self.H * 2, self.vocab_l * 4, 1 << 16)
            tpu.init_xgmi(self.device, slot_bytes)
        # prefill-sized all-reduces: RCCL async on its own stream,
        # overlapped with the next row-chunk's GEMM.  Needs the nccl(=RCCL)
        # backend; gloo (CPU CI) takes the inline path.
        import torch.distributed as dist
        self._async_ar = bool(
            self.world > 1 and dist.is_initialized()
            and "nccl" in str(dist.get_backend()).lower())

        self._upload_weights(weights)
        if max_seq is None:
            max_seq = self._auto_max_seq()
        self.max_seq = max_seq
        self._alloc_state(prefill_chunk)
        self._stack = self._native_stack()
        self._chains = self._decode_chains()
        self._graph = None
        self._graph_mode = None
        # side-stream weight prefetcher — measured NEGATIVE (the fork's
        # join makes the sequential prefetch chain the critical path:
        # fp8 1391 -> 764 tok/s), so off by default; LLM_PREFETCH=1 to
        # experiment
        import os as _os
        self.prefetch_on = _os.environ.get("LLM_PREFETCH", "0") == "1"
        self._pf_stream = torch.cuda.Stream(device=self.device)
        self._pf_sink = torch.zeros(256, dtype=torch.float32,
                                    device=self.device)
        self._pf_events = []
        self.launches_only = not (self.tp_branch or self.prefetch_on)

    # ------------------------------------------------------------------
    def _auto_max_seq(self) -> int:
        """KV pool length from free HBM (post-weights): fill the 288 GB
        MI355X budget instead of a fixed 4k default,
        capped at the model's max_position_embeddings."""
        cfg = self.config
        free, _total = torch.cuda.mem_get_info(self.device)
        esz = 1 if self.kv8 else 2
        per_pos = (cfg.num_hidden_layers * self.kvh_l * self.hd * 2 * esz
                   * self.max_batch)
        if self.kv8:
            per_pos += (cfg.num_hidden_layers * self.kvh_l * 2 * 4
                        * self.max_batch)  # scales
        per_pos += self.hd * 4 + 8  # rope tables + ring slot
        budget = int(free * 0.9) - (2 << 30)  # headroom for scratch/graph
        n = max(1024, budget // max(per_pos, 1))
        return int(min(cfg.max_position_embeddings, n))

    def _upload_weights(self, w: Dict[str, np.ndarray]):
        from ..io.loader import validate_weights

        validate_weights(self.config, w)  # actionable error vs KeyError
        cfg, dev = self.config, self.device
        tp, r = self.world, self.rank
        gemma = cfg.model_type == "gemma2"

        def bf16(a: np.ndarray) -> torch.Tensor:
            return torch.from_numpy(np.ascontiguousarray(a)).to(
                dev, torch.bfloat16, non_blocking=False)

        def gamma(a: np.ndarray) -> torch.Tensor:
            g = a.astype(np.float32) + (1.0 if gemma else 0.0)
            return torch.from_numpy(g).to(dev)

        def quant4(a: np.ndarray):
            """MXFP4: e2m1 packed 2/byte + e8m0 scale per 32 elems."""
            t = bf16(a)
            N, K = t.shape
            q = torch.empty(N, K // 2, dtype=torch.uint8, device=dev)
            e = torch.empty(N, K // 32, dtype=torch.uint8, device=dev)
            ho.quant_fp4(t, q, e)
            torch.cuda.synchronize()
            return q, e

        def quant8(a: np.ndarray):
            """Per-output-row e4m3fn quantization ON DEVICE (k_quant_
            fp8_rows): one bf16 upload, quantize, drop the bf16 copy —
            fp8 models hold a single weight copy in HBM and load in
            seconds (on the host 9B took ~90 s)."""
            t = bf16(a)
            N, K = t.shape
            q = torch.empty(N, K, dtype=torch.uint8, device=dev)
            s = torch.empty(N, dtype=torch.float32, device=dev)
            ho.quant_fp8(t, q, s)
            torch.cuda.synchronize()  # t freed right after
            return q, s

        self.embed = bf16(w["model.embed_tokens.weight"])
        lm_w = w.get("lm_head.weight", w["model.embed_tokens.weight"])
        if self.fp8:
            lmw = lm_w if tp == 1 else tpu.shard_rows(lm_w, r, tp)
            if self.keep_fp8:
                self.lm_head_q, self.lm_head_s = quant8(lmw)
            self.lm_head = None  # single-copy: no bf16 duplicate
            if self.wq4:
                self.lm_head_q4, self.lm_head_e4 = quant4(lmw)
        elif tp > 1:
            self.lm_head = bf16(tpu.shard_rows(lm_w, r, tp))
        elif lm_w is w.get("model.embed_tokens.weight", None) or \
                cfg.tie_word_embeddings and "lm_head.weight" not in w:
            self.lm_head = self.embed  # tied, share device memory
        else:
            self.lm_head = bf16(lm_w)
        self.g_final = gamma(w["model.norm.weight"])

        hd = cfg.head_dim
        self.layers = []
        for i in range(cfg.num_hidden_layers):
            p = f"model.layers.{i}"
            a = f"{p}.self_attn"
            hrows = lambda x: tpu.shard_rows(x, r, tp) if tp > 1 else x
            hcols = lambda x: tpu.shard_cols(x, r, tp) if tp > 1 else x
            import numpy as _np
            qkv_np = _np.concatenate([
                hrows(w[f"{a}.q_proj.weight"]),
                hrows(w[f"{a}.k_proj.weight"]),
                hrows(w[f"{a}.v_proj.weight"])], axis=0)
            if self.moe:
                # stacked per-expert [gate; up] rows (E*2I, H) and down
                # rows (E*H, I) — ONE device tensor per projection so the
                # decode GEMV can index expert e as a row offset
                # (eidx * 2I resp. eidx * H) off a device int32
                m = f"{p}.block_sparse_moe"
                E = cfg.num_local_experts
                gu_np = _np.concatenate(
                    [x for e in range(E)
                     for x in (w[f"{m}.experts.{e}.w1.weight"],
                               w[f"{m}.experts.{e}.w3.weight"])], axis=0)
                down_np = _np.concatenate(
                    [w[f"{m}.experts.{e}.w2.weight"] for e in range(E)],
                    axis=0)
            else:
                gu_np = _np.concatenate([
                    hrows(w[f"{p}.mlp.gate_proj.weight"]),
                    hrows(w[f"{p}.mlp.up_proj.weight"])], axis=0)
                down_np = hcols(w[f"{p}.mlp.down_proj.weight"])
            o_np = hcols(w[f"{a}.o_proj.weight"])
            lw = {
                "g_in": gamma(w[f"{p}.input_layernorm.weight"]),
                "g_post": gamma(w[f"{p}.post_attention_layernorm.weight"]),
            }
            if self.fp8:
                # SINGLE fp8 copy: decode GEMV and prefill fp8-MFMA GEMM
                # both read these (no bf16 duplicate in HBM)
                for name, arr in [("wqkv", qkv_np), ("wgu", gu_np),
                                  ("wo", o_np), ("wdown", down_np)]:
                    if self.keep_fp8:
                        lw[name + "_q"], lw[name + "_s"] = quant8(arr)
                    if self.wq4:
                        lw[name + "_q4"], lw[name + "_e4"] = quant4(arr)
            else:
                lw.update({"wqkv": bf16(qkv_np), "wgu": bf16(gu_np),
                           "wo": bf16(o_np), "wdown": bf16(down_np)})
            if self.moe:
                # router weights + decode-shaped views: the GEMV sees the
                # FIRST expert's rows (N=2I / N=H) and offsets the base
                # pointer by eidx * wstride device-side
                lw["wg"] = bf16(w[f"{p}.block_sparse_moe.gate.weight"])
                I2, H2 = 2 * self.inter_l, self.H
                if self.fp8:
                    lw["wgu_q_all"] = lw.pop("wgu_q")
                    lw["wgu_s_all"] = lw.pop("wgu_s")
                    lw["wdown_q_all"] = lw.pop("wdown_q")
                    lw["wdown_s_all"] = lw.pop("wdown_s")
                    lw["wgu_q"] = lw["wgu_q_all"][:I2]
                    lw["wgu_s"] = lw["wgu_s_all"][:I2]
                    lw["wdown_q"] = lw["wdown_q_all"][:H2]
                    lw["wdown_s"] = lw["wdown_s_all"][:H2]
                else:
                    lw["wgu_all"] = lw.pop("wgu")
                    lw["wdown_all"] = lw.pop("wdown")
                    lw["wgu"] = lw["wgu_all"][:I2]
                    lw["wdown"] = lw["wdown_all"][:H2]
            if gemma:
                lw["g_preffn"] = gamma(w[f"{p}.pre_feedforward_layernorm.weight"])
                lw["g_postffn"] = gamma(w[f"{p}.post_feedforward_layernorm.weight"])
            if cfg.attention_bias:
                # Qwen-2 family: fused qkv bias (decode GEMV adds it via
                # the res slot, the products of more rows as they store)
                bias_np = _np.concatenate([
                    hrows(w[f"{a}.q_proj.bias"]),
                    hrows(w[f"{a}.k_proj.bias"]),
                    hrows(w[f"{a}.v_proj.bias"])], axis=0)
                lw["bqkv"] = bf16(bias_np.reshape(1, -1))[0]
            self.layers.append(lw)

    def _alloc_state(self, prefill_chunk: int):
        cfg, dev = self.config, self.device
        S, hd = self.max_seq, self.hd
        L = cfg.num_hidden_layers
        bf = dict(dtype=torch.bfloat16, device=dev)
        kvt = torch.uint8 if self.kv8 else torch.bfloat16
        B = self.max_batch
        kv_shape = (self.kvh_l, S, hd) if B == 1 else (B, self.kvh_l, S, hd)
        self.k_cache = [torch.zeros(*kv_shape, dtype=kvt, device=dev)
                        for _ in range(L)]
        self.v_cache = [torch.zeros(*kv_shape, dtype=kvt, device=dev)
                        for _ in range(L)]
        if self.kv8:
            ks = (self.kvh_l, S) if B == 1 else (B, self.kvh_l, S)
            self.k_scale = [torch.zeros(*ks, dtype=torch.float32,
                                        device=dev) for _ in range(L)]
            self.v_scale = [torch.zeros(*ks, dtype=torch.float32,
                                        device=dev) for _ in range(L)]
        else:
            self.k_scale = [None] * L
            self.v_scale = [None] * L

        # RoPE tables fp32 (host-precomputed: guide App.B — no device trig)
        inv = cfg.rope_inv_freq()                      # (hd/2,) fp64
        t = np.arange(S, dtype=np.float64)
        freqs = np.outer(t, inv)
        self.cos_t = torch.from_numpy(np.cos(freqs).astype(np.float32)).to(dev)
        self.sin_t = torch.from_numpy(np.sin(freqs).astype(np.float32)).to(dev)

        # a group's prompts are read together
        PC = self.PC = min(prefill_chunk, max(256, self.max_seq * B))
        R = max(PC, self.max_batch)    # rows of a prompt's or a group's pass
        H, I = self.H, self.inter_l
        self.b_h = torch.zeros(R, H, **bf)
        self.b_xn = torch.zeros(R, H, **bf)
        self.b_t1 = torch.zeros(R, H, **bf)
        # q | k | v of a row, from one projection
        nqkv = (self.nh_l + 2 * self.kvh_l) * hd
        self.b_rqkv = torch.zeros(R, nqkv, **bf)
        self.b_att = torch.zeros(R, self.nh_l * hd, **bf)
        # act(gate) * up; of each of a row's experts
        pairs = R * (self.topk if self.moe else 1)
        self.b_gate = torch.zeros(pairs, I, **bf)
        # fp32 parts of products that split K, and of attention that splits
        # its keys.  A few long rows beside many outputs can take more than a
        # short chunk of a prompt does.
        few = [(nqkv, H), (H, self.nh_l * hd), (self.vocab_l, H)]
        if not self.moe:
            few += [(I, H, True), (H, I)]
        kinds = ["fp4"] * self.wq4 + ["fp8"] * self.keep_fp8 \
            if self.fp8 else ["bf16"]
        self.b_gemm_acc = torch.zeros(
            max([R * max(I, H)] +
                [ho.row_gemm_room(k, *p) for k in kinds for p in few]),
            dtype=torch.float32, device=dev)
        if self.fp8:
            # activation-quant scratch for the fp8 MFMA prefill GEMMs
            kmax = max(H, I, self.nh_l * hd)
            self.b_xq = torch.zeros(R * kmax, dtype=torch.uint8, device=dev)
            self.b_sx = torch.zeros(R, dtype=torch.float32, device=dev)
            if self.moe:
                self.b_aq = torch.zeros(pairs * I, dtype=torch.uint8,
                                        device=dev)
                self.b_sa = torch.zeros(pairs, dtype=torch.float32,
                                        device=dev)
            # act(gate) * up of few rows, to be rounded to e4m3 next
            self.b_act32 = torch.zeros(ho.FEW_ROWS, I, dtype=torch.float32,
                                       device=dev)
        # few-row products that split K: blocks that are done, by column
        # group (the parts go to b_gemm_acc)
        self.row_cnt = torch.zeros(256, dtype=torch.int32, device=dev)
        # the same of many-row products, by tile
        self.tile_cnt = torch.zeros(1024, dtype=torch.int32, device=dev)
        self.b_logits_l = torch.zeros(self.vocab_l, dtype=torch.float32,
                                      device=dev)
        self.b_logits = (self.b_logits_l if not self.tp_branch else
                         torch.zeros(cfg.vocab_size, dtype=torch.float32,
                                     device=dev))
        self.b_qkv = torch.zeros((self.nh_l + 2 * self.kvh_l) * hd, **bf)
        if self.moe:
            E = cfg.num_local_experts
            self.moe_idx = torch.zeros(R * self.topk, dtype=torch.int32,
                                       device=dev)
            self.moe_w = torch.zeros(R * self.topk, dtype=torch.float32,
                                     device=dev)
            self.moe_order = torch.zeros(pairs + 3 * (pairs // 32 + E),
                                         dtype=torch.int32, device=dev)
            self.b_pairs = torch.zeros(pairs, H, **bf)
        self.b_hb = torch.zeros(H, **bf)   # gemma residual ping-pong
        self.b_t2 = torch.zeros(H, **bf)   # gemma ffn-out delta
        # act(gate) * up of a decode step (of each expert): fp32 beside
        # weights that are multiplied in fp32
        self.b_act = torch.zeros(
            self.topk if self.moe else 1, I, device=dev,
            dtype=torch.float32 if self.fp8 else torch.bfloat16)
        # split-T decode attention scratch (partials + per-head tickets)
        import os as _os
        _sp = _os.environ.get("LLM_ATTN_SPLIT")
        # ranges of the history that a step may take: the kernel takes one
        # for some 256 keys (128 of 256 dims), up to so many
        self.attn_split = (int(_sp) if _sp else min(64, max(
            1, -(-self.max_seq // (128 if hd == 256 else 256)))))
        self.attn_scratch = torch.zeros(
            self.nh_l * self.attn_split * (hd + 2), dtype=torch.float32,
            device=dev)
        self.attn_cnt = torch.zeros(self.nh_l, dtype=torch.int32, device=dev)
        self.s_gmax = torch.zeros(1, dtype=torch.int64, device=dev)
        self.s_tops = torch.zeros(ho.CHAIN_TOPS, dtype=torch.float32,
                                  device=dev)
        self.s_pick = torch.zeros(1, dtype=torch.int64, device=dev)
        self.s_cnt = torch.zeros(1, dtype=torch.int32, device=dev)
        i32 = dict(dtype=torch.int32, device=dev)
        self.ids_buf = torch.zeros(PC, **i32)
        self.next_token = torch.zeros(1, **i32)
        self.out_ring = torch.zeros(max(65536, S + 16), **i32)
        self.nout = torch.zeros(1, **i32)
        self.len_buf = torch.zeros(1, **i32)
        self.rng_ctr = torch.zeros(1, dtype=torch.int64, device=dev)

        if self.max_batch > 1:
            B, nhh = self.max_batch, self.nh_l * hd
            # a chunk of several prompts: tokens, positions and pools of its
            # rows, the attention's tiles, the prompts' last rows
            pairs = PC * (self.nh_l // self.kvh_l)
            self.pack_buf = torch.zeros(
                3 * PC + 5 * (-(-pairs // 128) + B) + B, **i32)
            # the heads of its prompts, beside e4m3 weights
            self.b_row0 = torch.zeros(1, **i32)
            self.b_parts = torch.zeros(
                3 * ho.HEAD_ROWS * H if self.fp8 and not self.wq4 else 0, **bf)
            i64 = dict(dtype=torch.int64, device=dev)
            self.bt_qkv = self.b_rqkv[:B]
            self.bt_logits = torch.zeros(B, self.vocab_l, **bf)
            self.bt_logits32 = torch.zeros(B, cfg.vocab_size,
                                           dtype=torch.float32, device=dev)
            self.bt_next = torch.zeros(B, **i32)
            self.bt_lens = torch.zeros(B, **i32)  # ragged positions
            self.bt_ring = torch.zeros(B, S + 16, **i32)
            self.bt_nout = torch.zeros(B, **i32)
            self.bt_gmax = torch.zeros(B, **i64)
            self.bt_pick = torch.zeros(B, **i64)
            self.bt_cnt = torch.zeros(B, **i32)
            # for any number of active rows
            self.bt_scratch = torch.zeros(
                max(M * self._ranges(M) for M in range(1, B + 1)) *
                self.nh_l * (hd + 2), dtype=torch.float32, device=dev)
            self.bt_attn_cnt = torch.zeros(B * self.nh_l, **i32)
            # fused multi-x path scratch (fp8, B<=8)
            self.bt_gu = torch.zeros(B, 2 * I, **bf)
            self.bt_t1 = torch.zeros(B, H, **bf)
            self.bt_t2 = torch.zeros(B, H, **bf)
            self.bt_hb = torch.zeros(B, H, **bf)

        self.act = 0 if cfg.hidden_act == "silu" else 1
        self.gemma = cfg.model_type == "gemma2"
        self.attn_softcap = float(cfg.attn_logit_softcapping or 0.0)
        self.final_softcap = float(cfg.final_logit_softcapping or 0.0)
        self.scale = float(cfg.attn_scale)

    def _native_stack(self) -> ho.Stack:
        """The layers for the native launcher of a prompt's rows."""
        cfg = self.config

        def lin(lw, name):
            many = self.moe and name in ("wgu", "wdown")
            if self.wq4:
                return lw[name + "_q4"], None, lw[name + "_e4"]
            if self.fp8:
                end = "_all" if many else ""
                return lw[name + "_q" + end], lw[name + "_s" + end], None
            return lw[name + ("_all" if many else "")], None, None

        layers = []
        for i, lw in enumerate(self.layers):
            layers.append(dict(
                {n: lw.get(n) for n in ("g_in", "g_post", "g_preffn",
                                        "g_postffn", "bqkv", "wg")},
                qkv=lin(lw, "wqkv"), o=lin(lw, "wo"), gu=lin(lw, "wgu"),
                down=lin(lw, "wdown"), kc=self.k_cache[i],
                vc=self.v_cache[i], kS=self.k_scale[i], vS=self.v_scale[i],
                window=(cfg.sliding_window or 0) if cfg.is_sliding(i)
                else 0))
        own = {n: getattr(self, a, None) for n, a in dict(
            embed="embed", cos="cos_t", sin="sin_t", h="b_h", xn="b_xn",
            t1="b_t1", qkv="b_rqkv", att="b_att", gate="b_gate",
            acc="b_gemm_acc", row_cnt="row_cnt", tile_cnt="tile_cnt",
            xq="b_xq", sx="b_sx", len="len_buf", moe_idx="moe_idx",
            moe_w="moe_w", moe_order="moe_order", pairs="b_pairs",
            aq="b_aq", sa="b_sa").items()}
        return ho.Stack(
            layers, **own, acc_floats=self.b_gemm_acc.numel(),
            order_room=self.moe_order.numel() if self.moe else 0, H=self.H,
            I=self.inter_l, nh=self.nh_l, kvh=self.kvh_l, hd=self.hd,
            S=self.max_seq, wt=2 if self.wq4 else 1 if self.fp8 else 0,
            kv8=int(self.kv8), gemma=int(self.gemma), act=self.act,
            E=cfg.num_local_experts if self.moe else 0,
            topk=self.topk if self.moe else 0, nrow_cnt=self.row_cnt.numel(),
            ntile_cnt=self.tile_cnt.numel(),
            mfma=int(self.hd in (64, 128, 256)), rows=self.b_h.shape[0],
            pools=self.max_batch, eps=cfg.rms_norm_eps,
            scale=self.scale, softcap=self.attn_softcap,
            escale=cfg.embed_scale)

    def _decode_chains(self):
        """Of each layer the products behind its attention and those into the
        next one's, or the head, as one launch of a decode step; None where
        sizes or ranks do not let them be one.  What its products leave each
        other stands in chain_buf, a stretch of its own for every layer."""
        # its blocks are one a CU: with fewer CUs they would wait for turns
        cus = torch.cuda.get_device_properties(self.device) \
            .multi_processor_count
        if self.tp_branch or cus < ho.CHAIN_BLOCKS:
            return None
        H, I, n = self.H, self.inter_l, len(self.layers)
        act = self.b_act.dtype
        E, top = self.config.num_local_experts, self.topk if self.moe else 1
        if self.moe and (top > ho.CHAIN_TOP or E > ho.CHAIN_EXPERTS or
                         self.wq4):
            return None
        kinds = [(H, torch.bfloat16), (H, torch.bfloat16)] + \
            [(I, act)] * top + [(H, torch.float32)] * (top - 1)
        size = [ho.chain_room(*k) for k in kinds]
        each = sum(size) + ho.CHAIN_CLAIMS
        self.chain_buf = torch.zeros(n * each, dtype=torch.uint8,
                                     device=self.device)
        self.chain_h = torch.zeros(n, H, dtype=torch.bfloat16,
                                   device=self.device)

        def weight(lw, name):
            end = "_all" if self.moe and name in ("wgu", "wdown") else ""
            if self.wq4:
                return lw[name + "_q4"], None, lw[name + "_e4"]
            if self.fp8:
                return lw[name + "_q" + end], lw[name + "_s" + end], None
            return lw[name + end], None, None

        chains, h = [], self.b_h[0]
        for i, lw in enumerate(self.layers):
            at = i * each
            o, dn, *rest = (
                ho.chain_part(self.chain_buf, at + sum(size[:k]), *v)
                for k, v in enumerate(kinds))
            mid, part = rest[:top], rest[top:]
            gu = dict(W=weight(lw, "wgu"), x=o, y=mid[0], glu=True)
            down = dict(W=weight(lw, "wdown"), x=mid[-1], y=dn)
            st = [dict(W=weight(lw, "wo"), x=self.b_att[0], y=o), gu, down]
            if i + 1 < n:
                nxt = self.layers[i + 1]
                g_next = nxt["g_in"]
                last = dict(W=weight(nxt, "wqkv"), y=self.b_qkv,
                            add=nxt.get("bqkv"))
            else:
                g_next = self.g_final
                last = dict(W=weight(vars(self), "lm_head"), y=self.b_logits_l,
                            softcap=self.final_softcap, tops=self.s_tops)
            if self.gemma:
                gu.update(kind=ho.CHAIN_NORM2, h=h, g=lw["g_post"],
                          g2=lw["g_preffn"])
                h = self.chain_h[i]
                last.update(kind=ho.CHAIN_NORM2, g=lw["g_postffn"], g2=g_next,
                            hout=h)
            else:
                st[0].update(add=h)
                gu.update(kind=ho.CHAIN_NORM, g=lw["g_post"])
                down.update(add=o)
                last.update(kind=ho.CHAIN_NORM, g=g_next)
                h = dn
            if self.moe:
                # gate and up of each of a row's experts, then their sums
                gu.update(experts=E, slot=1)
                down.update(experts=E, slot=top, scaled=True)
                more = [dict(gu, slot=j + 1, y=mid[j]) for j in range(1, top)]
                gu.update(route=lw["wg"], top=top)
                sums = [dict(down, slot=j + 1, x=mid[j], y=part[j], add=None)
                        for j in range(top - 1)]
                if part:
                    down.update(add2=part[-1])
                st[2:] = more + sums + [down]
            chains.append(ho.Chain(st + [dict(x=dn, **last)],
                                   2 if self.wq4 else int(self.fp8),
                                   self.act, self.config.rms_norm_eps,
                                   self.chain_buf[at + sum(size):at + each]))
        return chains if all(c.fits() for c in chains) else None

    def _chunk_rows(self, n: int) -> int:
        """Rows of the chunks that a prompt of n tokens is read in."""
        return self.PC if self.tp_branch or n <= self.PC else \
            self._stack.chunk_rows(n, self.PC)

    def _read(self, ids: np.ndarray, pos0: int, layer_hook=None) -> None:
        """A chunk of a prompt (int32, up to PC tokens) from position pos0 of
        sequence _pb through all layers; its rows are in b_h."""
        M = len(ids)
        if M > ho.STACK_IDS:
            self.ids_buf[:M].copy_(torch.from_numpy(ids.astype(np.int32)))
            self._stack.embed(self.ids_buf, M, pos0)
        else:
            self._stack.embed(ids, M, pos0)
        self._layers_forward(M, layer_hook=layer_hook, keys=pos0 + M)

    # ------------------------------------------------------------------
    # cache interface (generate()-compatible)
    # ------------------------------------------------------------------
    def reset(self):
        self.len_buf.zero_()
        self.nout.zero_()
        self.rng_ctr.zero_()
        self.s_gmax.zero_()
        self.s_pick.zero_()
        self.s_cnt.zero_()
        self._host_len = 0  # host mirror of len_buf (overflow guard)

    # ------------------------------------------------------------------
    # layer stack over rows [0, M) of the scratch buffers
    # ------------------------------------------------------------------
    def _rows(self, lw, name, x, y, M: int, g=None, res=None, bias=None,
              act: int = -1, softcap: float = 0.0, batch: bool = False,
              ready: bool = False):
        """Projection of up to FEW_ROWS rows in one launch, W streamed
        once: norm of x (g; ``ready``: b_xq and b_sx hold the normed rows as
        e4m3), activation of gate and up rows (act), softcap, bias and
        residual on the way.  Rows beside e4m3 weights are rounded
        to e4m3, a row alone is not (GEMV).  ``batch``: a decode step of a
        group, which runs on the e4m3 copy where the engine holds MXFP4
        too."""
        eps = self.config.rms_norm_eps
        e4m3 = self.fp8 and (batch or not self.wq4)
        if e4m3 and M == 1:
            if g is not None:
                ho.rmsnorm(x[:1], g, self.b_xn[:1], eps=eps)
                x = self.b_xn
            assert bias is None or res is None, "one row adds one of them"
            ho.gemv_fp8(lw[name + "_q"], lw[name + "_s"], x, y,
                        res=res if bias is None else bias, softcap=softcap,
                        act=max(act, 0), glu=act >= 0)
            return
        if g is not None and not ready and x.shape[-1] > ho.ROW_NORM_K:
            if e4m3 and batch:
                ho.rmsnorm(x[:M], g, None, eps=eps, q2=self.b_xq,
                           s2=self.b_sx)
                ready = True
            else:
                ho.rmsnorm(x[:M], g, self.b_xn[:M], eps=eps)
                x, g = self.b_xn, None
        kw = dict(g=g, eps=eps, res=res, bias=bias, act=act, softcap=softcap,
                  part=self.b_gemm_acc, cnt=self.row_cnt)
        if e4m3:
            if g is None or ready:
                K, kw["g"] = x.shape[-1], None
                if not ready:
                    ho.quant_fp8(x[:M], self.b_xq, self.b_sx)
                x, kw["sx"] = self.b_xq[:M * K].view(M, K), self.b_sx
            # a prompt's rows are bf16 on their way to e4m3, a step's fp32
            ho.row_gemm(x, lw[name + "_q"], y, M, ws=lw[name + "_s"],
                        norm16=not batch, **kw)
        elif self.wq4:
            ho.row_gemm(x, lw[name + "_q4"], y, M, we=lw[name + "_e4"], **kw)
        else:
            ho.row_gemm(x, lw[name], y, M, **kw)

    def _linear(self, lw, name, x, y, res=None, M: int = 1,
                batch: bool = False, bias=None, act: int = -1):
        """Projection by weight NAME so dtype routing stays in one
        place: few rows, bf16 MFMA GEMM, or (fp8) fp8-MFMA GEMM with
        on-the-fly activation row quantization.  ``act``: gate and up rows,
        y = act(gate) * up."""
        if M <= ho.FEW_ROWS:
            self._rows(lw, name, x, y, M, res=res, bias=bias, act=act,
                       batch=batch)
            return
        res = res[:M] if res is not None else None
        kw = dict(res=res, accbuf=self.b_gemm_acc, bias=bias, act=act,
                  cnt=self.tile_cnt)
        if self.wq4:
            assert act < 0 or res is None, "a gate beside MXFP4 adds nothing"
            ho.gemm_fp4w(x[:M], lw[name + "_q4"], lw[name + "_e4"], y[:M],
                         **kw)
            return
        if self.fp8:
            ho.quant_fp8(x[:M], self.b_xq, self.b_sx)
            ho.gemm_fp8(self.b_xq, self.b_sx, lw[name + "_q"],
                        lw[name + "_s"], y[:M], M, x.shape[-1], **kw)
        else:
            ho.gemm(x[:M], lw[name], y, **kw)

    def _rowpar_ar(self, lw, name, x, y, M: int, batch: bool = False):
        """Row-parallel projection followed by all-reduce over TP ranks.
        For prefill-sized M the rows are split in two: the all-reduce of
        chunk A runs on RCCL's comm stream while chunk B's GEMM occupies
        the compute stream (the reference has no distributed code at
        all)."""
        if not (self._async_ar and M >= 512):
            self._linear(lw, name, x, y, M=M, batch=batch)
            tpu.all_reduce(y[:M])
            return
        import torch.distributed as dist
        K = x.shape[-1]
        if self.fp8 and not self.wq4:
            ho.quant_fp8(x[:M], self.b_xq, self.b_sx)
        works = []
        M2 = M // 2
        for a, b in ((0, M2), (M2, M)):
            if self.wq4:
                ho.gemm_fp4w(x[a:b], lw[name + "_q4"], lw[name + "_e4"],
                             y[a:b], accbuf=self.b_gemm_acc,
                             cnt=self.tile_cnt)
            elif self.fp8:
                ho.gemm_fp8(self.b_xq[a * K:], self.b_sx[a:],
                            lw[name + "_q"], lw[name + "_s"], y[a:b],
                            b - a, K, accbuf=self.b_gemm_acc,
                            cnt=self.tile_cnt)
            else:
                ho.gemm(x[a:b], lw[name], y[a:b], accbuf=self.b_gemm_acc,
                        cnt=self.tile_cnt)
            # async -> lands on the RCCL stream after the chunk's GEMM;
            # the compute stream proceeds to the next chunk immediately
            works.append(dist.all_reduce(y[a:b], async_op=True))
        for wk in works:
            wk.wait()  # compute stream waits on the comm stream

    def _kc(self, i):
        return self.k_cache[i] if self.max_batch == 1 else \
            self.k_cache[i][self._pb]

    def _vc(self, i):
        return self.v_cache[i] if self.max_batch == 1 else \
            self.v_cache[i][self._pb]

    def _ks(self, i):
        s = self.k_scale[i]
        return s if (s is None or self.max_batch == 1) else s[self._pb]

    def _vs(self, i):
        s = self.v_scale[i]
        return s if (s is None or self.max_batch == 1) else s[self._pb]

    def _ranges(self, M: int) -> int:
        """Ranges of the history that a step of M rows may take: the more
        rows, the fewer fill the chip.  us, 8000 keys of 8 heads of 128, by
        1, 2, 4, 8, 16 ranges: one row 80 47 28 19 15, four 103 61 37 32 31,
        16 127 99 102 102 103; 16 rows of 620 keys, 8 heads of 256: one range
        25, two 23, three 30.  A block of 256 dims is all that a CU holds, so
        there each four query heads of a kv head count: 16 rows of 109 and 2031
        keys, 8/1 heads, by 8 ranges 9.8 and 22, by 16 17 and 30."""
        blocks = M * self.kvh_l
        if self.hd == 256:
            blocks *= -(-self.nh_l // (4 * self.kvh_l))
        return min(self.attn_split, max(1, 256 // blocks))

    def _layers_forward(self, M: int, layer_hook=None,
                        batch_attn: bool = False, keys: int = 0, pack=None):
        """Layer stack over rows [0, M), the last of which sees ``keys``
        keys.  ``pack``: rows of several prompts, (rows, tiles, longest) of
        `_read_pack`.  ``batch_attn``: rows are M
        INDEPENDENT sequences at the same position (lockstep batched
        decode) — the fused decode-attention kernel runs per row over
        per-sequence KV pools instead of the prefill attention."""
        if not batch_attn and not self.tp_branch:
            rows, tiles, most = pack or (None, None, 0)
            kw = dict(keys=keys, pool=self._pb, rows=rows, tiles=tiles,
                      most=most)
            if layer_hook is None:
                self._stack.forward(M, **kw)
                return
            layer_hook(-1, self.b_h[:M])
            for i in range(len(self.layers)):
                self._stack.forward(M, first=i, last=i + 1, **kw)
                layer_hook(i, self.b_h[:M])
            return
        self._layers_by_launch(M, layer_hook, batch_attn, keys, pack)

    def _layers_by_launch(self, M: int, layer_hook=None,
                          batch_attn: bool = False, keys: int = 0, pack=None):
        """The same with a call a launch: steps of a group (captured once)
        and layers that reduce over ranks in between."""
        cfg = self.config
        eps = cfg.rms_norm_eps
        h, xn, t1 = self.b_h, self.b_xn, self.b_t1
        few = M <= ho.FEW_ROWS
        # a step's rows go from one norm to the next as e4m3 (Gemma)
        step8 = self.gemma and few and batch_attn and self.fp8 and M > 1
        qkv = self.b_rqkv[:M]
        nq, nkv = self.nh_l * self.hd, self.kvh_l * self.hd
        q, k, v = qkv.split([nq, nkv, nkv], dim=1)

        def into_h(name, x, g=None):
            """h += x W^T (over all ranks), Gemma's through its post norm
            and, with g, on to the norm that follows."""
            post = {"wo": "g_post", "wdown": "g_postffn"}[name]
            if self.gemma:
                self._rowpar_ar(lw, name, x, t1, M, batch_attn)
                to = {} if g is None else \
                    dict(g2=g, q2=self.b_xq, s2=self.b_sx) if step8 else \
                    dict(g2=g, y2=xn[:M])
                ho.rmsnorm(t1[:M], lw[post], h[:M], res=h[:M], eps=eps, **to)
            elif self.tp_branch:
                self._rowpar_ar(lw, name, x, t1, M, batch_attn)
                ho.addinto(h[:M], t1[:M])
            else:
                self._linear(lw, name, x, h, res=h, M=M, batch=batch_attn)

        if layer_hook is not None:
            layer_hook(-1, h[:M])  # embedding output
        for i, lw in enumerate(self.layers):
            window = cfg.sliding_window if cfg.is_sliding(i) else 0
            if few:
                self._rows(lw, "wqkv", h, qkv, M, g=lw["g_in"],
                           bias=lw.get("bqkv"), batch=batch_attn,
                           ready=step8 and i > 0)
            else:
                if not self.gemma or i == 0:    # else by the layer before
                    ho.rmsnorm(h[:M], lw["g_in"], xn[:M], eps=eps)
                self._linear(lw, "wqkv", xn, qkv, M=M, bias=lw.get("bqkv"))
            if batch_attn:
                ho.attn_dec(qkv, self.k_cache[i], self.v_cache[i],
                            self.b_att[0], self.bt_lens, self.cos_t,
                            self.sin_t, self.bt_scratch, self.bt_attn_cnt,
                            self.nh_l, self.kvh_l, self.hd, self.scale,
                            softcap=self.attn_softcap, window=window or 0,
                            split=self._ranges(M), kS=self.k_scale[i],
                            vS=self.v_scale[i], batch=M)
            elif pack is not None:
                rows, tiles, most = pack
                kv = dict(kS=self.k_scale[i], vS=self.v_scale[i])
                ho.rope_cache(q, k, v, self.k_cache[i], self.v_cache[i],
                              self.cos_t, self.sin_t, self.len_buf, M,
                              self.nh_l, self.kvh_l, self.hd, rows=rows, **kv)
                ho.attn_prefill_mfma(
                    q, self.k_cache[i], self.v_cache[i], self.b_att,
                    self.len_buf, M, self.nh_l, self.kvh_l, self.hd,
                    self.scale, softcap=self.attn_softcap, window=window or 0,
                    part=self.b_gemm_acc, keys=keys, tiles=tiles, most=most,
                    **kv)
            else:
                ho.rope_cache(q, k, v, self._kc(i),
                              self._vc(i), self.cos_t, self.sin_t,
                              self.len_buf, M, self.nh_l, self.kvh_l,
                              self.hd, kS=self._ks(i), vS=self._vs(i))
                if self.hd in (64, 128, 256):
                    ho.attn_prefill_mfma(
                        q, self._kc(i), self._vc(i), self.b_att,
                        self.len_buf, M, self.nh_l, self.kvh_l, self.hd,
                        self.scale, softcap=self.attn_softcap,
                        window=window or 0,
                        kS=self._ks(i), vS=self._vs(i),
                        part=self.b_gemm_acc, keys=keys)
                else:
                    # per-query VALU kernel: every production head_dim is
                    # 64/128/256 (MFMA above); kept as the documented
                    # debugging/odd-shape fallback
                    ho.attn(q, self._kc(i), self._vc(i),
                            self.b_att, self.len_buf, M, self.nh_l,
                            self.kvh_l, self.hd, self.scale,
                            softcap=self.attn_softcap,
                            window=window or 0,
                            kS=self._ks(i), vS=self._vs(i))
            g_mlp = lw["g_preffn"] if self.gemma else lw["g_post"]
            into_h("wo", self.b_att, g_mlp if step8 or not few else None)
            if self.moe:
                ho.rmsnorm(h[:M], g_mlp, xn[:M], eps=eps)
                self._moe_mlp_rows(lw, M)
            else:
                a = self.b_gate
                if few:
                    if 1 < M and self.fp8 and batch_attn:
                        a = self.b_act32
                    self._rows(lw, "wgu", h, a, M, g=g_mlp, act=self.act,
                               batch=batch_attn, ready=step8)
                else:
                    if not self.gemma:
                        ho.rmsnorm(h[:M], g_mlp, xn[:M], eps=eps)
                    self._linear(lw, "wgu", xn, a, M=M, act=self.act)
                last = few and not step8 or i + 1 == len(self.layers)
                into_h("wdown", a,
                       None if last else self.layers[i + 1]["g_in"])
            if layer_hook is not None:
                layer_hook(i, h[:M])

    def _moe_mlp_rows(self, lw, M: int):
        """Prefill/batch MoE MLP over rows [0, M): the router's choices,
        sorted by expert on the device, then both products over each
        expert's own rows, and a row's results weighted into h; decode
        multiplies by the chosen experts directly (`_decode_step`)."""
        cfg = self.config
        E, I, H, top = (cfg.num_local_experts, self.inter_l, self.H,
                        self.topk)
        pairs = M * top
        a, order = self.b_gate[:pairs], self.moe_order
        ho.moe_route(self.b_h, lw["g_post"], lw["wg"], M, top,
                     self.moe_idx, self.moe_w, eps=cfg.rms_norm_eps)
        ho.expert_sort(self.moe_idx, order, pairs, E)
        if self.fp8:
            ho.quant_fp8(self.b_xn[:M], self.b_xq, self.b_sx)
            ho.expert_gemm(self.b_xq, lw["wgu_q_all"], a, order, pairs, E,
                           top, H, True, act=self.act, sx=self.b_sx,
                           sw=lw["wgu_s_all"])
            ho.quant_fp8(a, self.b_aq, self.b_sa)
            ho.expert_gemm(self.b_aq, lw["wdown_q_all"], self.b_pairs, order,
                           pairs, E, top, I, False, sx=self.b_sa,
                           sw=lw["wdown_s_all"])
        else:
            ho.expert_gemm(self.b_xn, lw["wgu_all"], a, order, pairs, E, top,
                           H, True, act=self.act)
            ho.expert_gemm(a, lw["wdown_all"], self.b_pairs, order, pairs, E,
                           top, I, False)
        ho.expert_sum(self.b_pairs, self.moe_w, self.moe_idx, self.b_h, M,
                      top)

    @property
    def _head(self):
        """lm_head under the weight names that _rows expects."""
        if self.fp8:
            h = {"_q4": self.lm_head_q4, "_e4": self.lm_head_e4} \
                if self.wq4 else {}
            if self.keep_fp8:
                h.update({"_q": self.lm_head_q, "_s": self.lm_head_s})
            return h
        return {"": self.lm_head}

    def _head_rows(self, M: int, out: torch.Tensor, batch: bool = False):
        """out[:M] = logits (bf16, this rank's vocabulary) of rows of h."""
        if M <= ho.FEW_ROWS:
            self._rows(self._head, "", self.b_h, out, M, g=self.g_final,
                       softcap=self.final_softcap, batch=batch)
            return
        ho.rmsnorm(self.b_h[:M], self.g_final, self.b_xn[:M],
                   eps=self.config.rms_norm_eps)
        if self.wq4 and not batch:
            ho.gemm_fp4w(self.b_xn[:M], self.lm_head_q4, self.lm_head_e4,
                         out[:M], accbuf=self.b_gemm_acc,
                         cnt=self.tile_cnt)
        elif self.fp8:
            ho.quant_fp8(self.b_xn[:M], self.b_xq, self.b_sx)
            ho.gemm_fp8(self.b_xq, self.b_sx, self.lm_head_q, self.lm_head_s,
                        out[:M], M, self.H, accbuf=self.b_gemm_acc,
                        cnt=self.tile_cnt)
        else:
            ho.gemm(self.b_xn[:M], self.lm_head, out[:M],
                    accbuf=self.b_gemm_acc, cnt=self.tile_cnt)
        if self.final_softcap:
            ho.softcap(out[:M], self.final_softcap)

    def _lm_head_last(self, M: int):
        """Final norm + lm_head on row M - 1 -> self.b_logits (f32, V);
        the norm rides in the GEMV staging pass (no separate launch)."""
        hrow = self.b_h[M - 1]
        kw = dict(stage=ho.STAGE_NORM, g=self.g_final,
                  eps=self.config.rms_norm_eps, softcap=self.final_softcap)
        if self.wq4:
            ho.gemv_fp4(self.lm_head_q4, self.lm_head_e4, hrow,
                        self.b_logits_l, **kw)
        elif self.fp8:
            ho.gemv_fp8(self.lm_head_q, self.lm_head_s, hrow,
                        self.b_logits_l, **kw)
        else:
            ho.gemv(self.lm_head, hrow, self.b_logits_l, **kw)
        if self.tp_branch:
            tpu.all_gather_into(self.b_logits, self.b_logits_l)

    def forward_full(self, ids: np.ndarray,
                     return_hidden_states: bool = False):
        """All-positions logits (M, V) — reference-parity API (the HF
        tuple shape).  Prefill-style pass; vocab GEMM per
        chunk.  Resets the cache.  With ``return_hidden_states`` also
        returns the L+1 per-layer hidden states (embedding output +
        each decoder layer, reference ``all_hidden_states``
        llama3.2_model.py:682-716) as fp32 numpy arrays."""
        ids = np.asarray(ids, dtype=np.int32).ravel()
        self.reset()
        if not return_hidden_states:
            return self.forward_positions(ids, 0)
        n = len(ids)
        out = np.empty((n, self.config.vocab_size), dtype=np.float32)
        L = self.config.num_hidden_layers
        hidden = [np.empty((n, self.H), dtype=np.float32)
                  for _ in range(L + 1)]
        logits_buf = torch.empty(self.PC, self.vocab_l,
                                 dtype=torch.bfloat16, device=self.device)
        done = 0
        while done < n:
            M = min(n - done, self.PC)
            d0 = done

            def hook(i, h):
                torch.cuda.synchronize()
                hidden[i + 1][d0:d0 + h.shape[0]] = \
                    h.float().cpu().numpy()
            self._read(ids[done:done + M], done, layer_hook=hook)
            self._head_rows(M, logits_buf)
            if self.world > 1:
                # gather vocab shards on-device (each rank holds the
                # columns [r*vocab_l, (r+1)*vocab_l) of rows [0, M))
                import torch.distributed as dist
                t = logits_buf[:M].float().contiguous()
                chunks = [torch.empty_like(t) for _ in range(self.world)]
                dist.all_gather(chunks, t)
                loc = torch.cat(chunks, dim=1).cpu().numpy()
            else:
                torch.cuda.synchronize()
                loc = logits_buf[:M].float().cpu().numpy()
            out[done:done + M] = loc
            done += M
        ho.i32_set(self.len_buf, n)
        # mirror the device len so a following decode()'s overflow guard
        # counts from the right base (it would run past the pool otherwise)
        self._host_len = n
        if return_hidden_states:
            return out, hidden
        return out

    def forward_positions(self, ids: np.ndarray, pos0: int) -> np.ndarray:
        """All-position logits (M, V) fp32, CONTINUING from pos0 (no
        cache reset: KV for ids lands at [pos0, pos0+M) and the pool can
        be rolled back afterwards with ``rewind``).  This is the
        speculative-decoding VERIFY pass: the target model scores k
        draft tokens in one prefill-shaped pass instead of k decode
        steps (the reference has nothing comparable)."""
        ids = np.asarray(ids, dtype=np.int32).ravel()
        n = len(ids)
        if n == 0:
            raise ValueError("empty ids")
        if pos0 + n > self.max_seq:
            raise ValueError(f"sequence {pos0}+{n} exceeds max_seq "
                             f"{self.max_seq}")
        out = None
        logits_buf = torch.empty(min(n, self.PC), self.vocab_l,
                                 dtype=torch.bfloat16, device=self.device)
        done = 0
        rows = self._chunk_rows(n)
        while done < n:
            M = min(n - done, rows)
            self._read(ids[done:done + M], pos0 + done)
            self._head_rows(M, logits_buf)
            if done + M == n:
                ho.i32_set(self.len_buf, pos0 + n)
                self._host_len = pos0 + n
            if self.world > 1:
                # gather vocab shards on-device (each rank holds the
                # columns [r*vocab_l, (r+1)*vocab_l) of rows [0, M))
                import torch.distributed as dist
                t = logits_buf[:M].float().contiguous()
                chunks = [torch.empty_like(t) for _ in range(self.world)]
                dist.all_gather(chunks, t)
                loc = torch.cat(chunks, dim=1).cpu().numpy()
            else:
                loc = logits_buf[:M].float().cpu().numpy()
            if M == n:           # widened on the device, copied once
                return loc
            if out is None:
                out = np.empty((n, self.config.vocab_size), dtype=np.float32)
            out[done:done + M] = loc
            done += M
        return out

    def rewind(self, n: int):
        """Roll the sequence back to length n — O(1): the KV pool is
        preallocated and the attention kernels read the device length
        from len_buf, so positions >= n are dead until overwritten.
        Speculative decoding uses this to discard rejected draft KV."""
        if not 0 <= n <= self.max_seq:
            raise ValueError(f"rewind {n} outside [0, {self.max_seq}]")
        ho.i32_set(self.len_buf, n)
        self._host_len = n

    # ------------------------------------------------------------------
    # generic forward (oracle-parity / generate()-compatible)
    # ------------------------------------------------------------------
    def forward(self, ids: np.ndarray, cache: DeviceCacheHandle,
                pos0: int) -> np.ndarray:
        """Returns last-position logits (1, V) fp32 numpy."""
        ids = np.asarray(ids, dtype=np.int32).ravel()
        if pos0 != cache.seq_len:
            raise ValueError("GPU engine requires sequential positions")
        n = len(ids)
        if n == 0:
            raise ValueError("empty ids")
        if pos0 + n > self.max_seq:
            raise ValueError(f"sequence {pos0}+{n} exceeds max_seq "
                             f"{self.max_seq}")
        done = 0
        rows = self._chunk_rows(n)
        while done < n:
            M = min(n - done, rows)
            self._read(ids[done:done + M], pos0 + done)
            done += M
        self._lm_head_last(M)
        ho.i32_set(self.len_buf, pos0 + n)
        self._host_len = pos0 + n
        cache.seq_len = pos0 + n
        return self.b_logits.cpu().numpy()[None, :]     # waits for it

    # ------------------------------------------------------------------
    # fast device-side decode loop (graph-replayable)
    # ------------------------------------------------------------------
    def _dgemv(self, lw, name, x, y, **kw):
        """Decode GEMV: MXFP4 / fp8 / bf16 weights by engine dtype."""
        if self.wq4:
            ho.gemv_fp4(lw[name + "_q4"], lw[name + "_e4"], x, y, **kw)
        elif self.fp8:
            ho.gemv_fp8(lw[name + "_q"], lw[name + "_s"], x, y, **kw)
        else:
            ho.gemv(lw[name], x, y, **kw)

    def _pf_tensors(self, lw):
        if self.wq4:
            return (lw["wqkv_q4"], lw["wo_q4"], lw["wgu_q4"],
                    lw["wdown_q4"])
        if self.fp8:
            return (lw["wqkv_q"], lw["wo_q"], lw["wgu_q"], lw["wdown_q"])
        return (lw["wqkv"], lw["wo"], lw["wgu"], lw["wdown"])

    def _decode_step(self, greedy: bool, min_p: float,
                     temperature: float = 1.0):
        """Fused decode path: 2 kernels a layer where its products, and with
        the last layer's the head, run as one launch (``_decode_chains``),
        else 5 — RMSNorm lives in the staging of a product, GLU in the
        epilogue of gate and up, RoPE + KV write inside the attention kernel;
        a side stream prefetches the next layer's weights through MALL, paced
        by per-layer events."""
        cfg = self.config
        eps = cfg.rms_norm_eps
        h = self.b_h[0]
        hnext = self.b_hb
        t1 = self.b_t1[0]
        t2 = self.b_t2
        s0 = torch.cuda.current_stream()
        pf = self.prefetch_on
        chains = None if pf else self._chains
        # what the chains' products leave each other is not there yet
        ones = dict(ones=self.chain_buf) if chains else {}
        self._pf_events = []
        prev = None  # previous gemma layer (its postffn norm fused here)
        for i, lw in enumerate(self.layers):
            if pf and i + 1 < len(self.layers):
                ev = torch.cuda.Event()
                ev.record(s0)
                self._pf_events.append(ev)
                self._pf_stream.wait_event(ev)
                with torch.cuda.stream(self._pf_stream):
                    for t in self._pf_tensors(self.layers[i + 1]):
                        ho.prefetch(t, self._pf_sink)
            window = cfg.sliding_window if cfg.is_sliding(i) else 0
            if chains and i > 0:
                pass                      # with the layer before
            elif self.gemma and prev is not None:
                # h' = h + norm(t2_prev)*g_postffn_prev; stage norm(h')*g_in
                self._dgemv(lw, "wqkv", t2, self.b_qkv,
                            stage=ho.STAGE_NORM2, x2=h,
                            g=prev["g_postffn"], g2=lw["g_in"], res=hnext,
                            eps=eps)
                h, hnext = hnext, h
            elif i == 0 and "bqkv" not in lw:
                # layer 0: embed gather fused into the QKV staging pass
                # (x = table, x2 = sampled token id, res = persisted h)
                self._dgemv(lw, "wqkv", self.embed, self.b_qkv,
                            stage=ho.STAGE_NORM_EMBED, x2=self.next_token,
                            g=lw["g_in"], res=h, eps=eps,
                            escale=cfg.embed_scale, **ones)
            else:
                if i == 0:  # bias models keep the separate embed gather
                    ho.embed(self.embed, self.next_token, self.b_h, 1,
                             cfg.embed_scale)
                self._dgemv(lw, "wqkv", h, self.b_qkv, stage=ho.STAGE_NORM,
                            g=lw["g_in"], res=lw.get("bqkv"), eps=eps, **ones)
            prev = lw
            ho.attn_dec(self.b_qkv, self.k_cache[i], self.v_cache[i],
                        self.b_att[0], self.len_buf, self.cos_t, self.sin_t,
                        self.attn_scratch, self.attn_cnt,
                        self.nh_l, self.kvh_l, self.hd, self.scale,
                        softcap=self.attn_softcap, window=window or 0,
                        split=self.attn_split,
                        kS=self.k_scale[i], vS=self.v_scale[i])
            if chains:
                chains[i].run()
                continue
            if self.gemma:
                self._dgemv(lw, "wo", self.b_att[0], t1)
                tpu.all_reduce(t1)
                # NORM2: h' = h + norm(t1)*g_post (persisted to hnext),
                # stage = norm(h')*g_preffn — both sandwich norms fused
                self._dgemv(lw, "wgu", t1, self.b_act, stage=ho.STAGE_NORM2,
                            x2=h, g=lw["g_post"], g2=lw["g_preffn"],
                            res=hnext, eps=eps, glu=True, act=self.act)
                h, hnext = hnext, h
                self._dgemv(lw, "wdown", self.b_act, t2)
                tpu.all_reduce(t2)
            else:
                if self.tp_branch:
                    self._dgemv(lw, "wo", self.b_att[0], t1)
                    tpu.all_reduce(t1)
                    ho.addinto(h, t1)
                else:
                    self._dgemv(lw, "wo", self.b_att[0], h, res=h)
                if self.moe:
                    # router -> both products of all topk experts at once:
                    # W by the device's idx, the second one's results
                    # weighted by the device's router probs into h
                    ho.moe_route(h, lw["g_post"], lw["wg"], 1, self.topk,
                                 self.moe_idx, self.moe_w, eps=eps)
                    I, H = self.inter_l, self.H
                    ei = self.moe_idx[:self.topk]
                    up = dict(stage=ho.STAGE_NORM, g=lw["g_post"], eps=eps,
                              glu=True, act=self.act, eidx=ei,
                              wstride=2 * I * H)
                    dn = dict(res=h, eidx=ei, wstride=H * I,
                              oscale=self.moe_w)
                    if self.fp8:
                        ho.gemv_fp8(lw["wgu_q"], lw["wgu_s"], h, self.b_act,
                                    sstride=2 * I, **up)
                        ho.gemv_fp8(lw["wdown_q"], lw["wdown_s"], self.b_act,
                                    h, sstride=H, **dn)
                    else:
                        ho.gemv(lw["wgu"], h, self.b_act, **up)
                        ho.gemv(lw["wdown"], self.b_act, h, **dn)
                    continue
                self._dgemv(lw, "wgu", h, self.b_act, stage=ho.STAGE_NORM,
                            g=lw["g_post"], eps=eps, glu=True, act=self.act)
                if self.tp_branch:
                    self._dgemv(lw, "wdown", self.b_act, t1)
                    tpu.all_reduce(t1)
                    ho.addinto(h, t1)
                else:
                    self._dgemv(lw, "wdown", self.b_act, h, res=h)
        if pf:
            ev = torch.cuda.Event()
            ev.record(self._pf_stream)
            self._pf_events.append(ev)
            s0.wait_event(ev)  # join the fork before the step ends
        if chains:
            pass                          # the head with the last layer
        elif self.gemma:
            # last layer's post-ffn sandwich norm + final norm, both
            # fused into the lm_head staging (NORM2: h' = h + norm(t2)*
            # g_postffn, then stage norm(h')*g_final)
            kw = dict(stage=ho.STAGE_NORM2, x2=h,
                      g=self.layers[-1]["g_postffn"], g2=self.g_final,
                      res=hnext, eps=eps, softcap=self.final_softcap)
            if self.wq4:
                ho.gemv_fp4(self.lm_head_q4, self.lm_head_e4, t2,
                            self.b_logits_l, **kw)
            elif self.fp8:
                ho.gemv_fp8(self.lm_head_q, self.lm_head_s, t2,
                            self.b_logits_l, **kw)
            else:
                ho.gemv(self.lm_head, t2, self.b_logits_l, **kw)
        else:
            # final norm fused into the lm_head staging pass
            kw = dict(stage=ho.STAGE_NORM, g=self.g_final, eps=eps,
                      softcap=self.final_softcap)
            if self.wq4:
                ho.gemv_fp4(self.lm_head_q4, self.lm_head_e4, h,
                            self.b_logits_l, **kw)
            elif self.fp8:
                ho.gemv_fp8(self.lm_head_q, self.lm_head_s, h,
                            self.b_logits_l, **kw)
            else:
                ho.gemv(self.lm_head, h, self.b_logits_l, **kw)
        if self.tp_branch:
            tpu.all_gather_into(self.b_logits, self.b_logits_l)
        ho.sample(self.b_logits, min_p, greedy, self.seed, self.rng_ctr,
                  self.s_gmax, self.s_pick, self.next_token, self.out_ring,
                  self.nout, self.len_buf, bump_len=True,
                  temperature=temperature, cnt=self.s_cnt,
                  tops=self.s_tops if chains else None)

    # ------------------------------------------------------------------
    # lockstep batched decode (throughput mode; beyond-parity capability)
    # ------------------------------------------------------------------
    def _decode_batch_step(self, B: int, greedy: bool, min_p: float,
                           temperature: float = 1.0):
        """One decode step for B lockstep sequences: the layer stack over
        B rows, up to FEW_ROWS of them with W streamed once a projection.
        Graph-replayable (all state device-side).  The multi-x GEMV path
        (fp8, B<=8, VALU-bound) is there for comparison, by
        LLM_BATCH_MX_MAX."""
        cfg = self.config
        import os as _os  # noqa: delayed so env changes apply per call
        mx_max = int(_os.environ.get("LLM_BATCH_MX_MAX", "0"))
        if (self.fp8 and B <= mx_max and not cfg.attention_bias
                and not self.moe):
            return self._decode_batch_step_mx(B, greedy, min_p, temperature)
        ho.embed(self.embed, self.bt_next, self.b_h, B, cfg.embed_scale)
        self._layers_forward(B, batch_attn=True)
        self._head_rows(B, self.bt_logits, batch=True)
        ho.sample(self.bt_logits[:B], min_p, greedy, self.seed,
                  self.rng_ctr, self.bt_gmax, self.bt_pick, self.bt_next,
                  self.bt_ring, self.bt_nout, self.bt_lens, bump_len=True,
                  temperature=temperature, cnt=self.bt_cnt, batch=B)

    def _decode_batch_step_mx(self, B: int, greedy: bool, min_p: float,
                              temperature: float = 1.0):
        """Fused batched decode (fp8, B<=8): mirrors _decode_step's
        kernels with multi-x GEMVs over B rows."""
        cfg = self.config
        eps = cfg.rms_norm_eps
        H, I = self.H, self.inter_l
        h = self.b_h            # rows 0..B = per-seq h
        hb = self.bt_hb         # gemma ping-pong
        t1, t2, gu = self.bt_t1, self.bt_t2, self.bt_gu
        qkvw = (self.nh_l + 2 * self.kvh_l) * self.hd
        nhh = self.nh_l * self.hd
        prev = None
        for i, lw in enumerate(self.layers):
            window = cfg.sliding_window if cfg.is_sliding(i) else 0
            if self.gemma and prev is not None:
                ho.gemv_fp8_mx(lw["wqkv_q"], lw["wqkv_s"], t2, self.bt_qkv,
                               B, H, qkvw, stage=ho.STAGE_NORM2, x2=h,
                               x2stride=H, g=prev["g_postffn"],
                               g2=lw["g_in"], hout=hb, hstride=H, eps=eps)
                h, hb = hb, h
            elif i == 0:
                ho.gemv_fp8_mx(lw["wqkv_q"], lw["wqkv_s"], self.embed,
                               self.bt_qkv, B, 0, qkvw,
                               stage=ho.STAGE_NORM_EMBED,
                               x2=self.bt_next, g=lw["g_in"], hout=h,
                               hstride=H, eps=eps,
                               escale=cfg.embed_scale)
            else:
                ho.gemv_fp8_mx(lw["wqkv_q"], lw["wqkv_s"], h, self.bt_qkv,
                               B, H, qkvw, stage=ho.STAGE_NORM,
                               g=lw["g_in"], eps=eps)
            prev = lw
            ho.attn_dec(self.bt_qkv, self.k_cache[i], self.v_cache[i],
                        self.b_att[0], self.bt_lens, self.cos_t, self.sin_t,
                        self.bt_scratch, self.bt_attn_cnt,
                        self.nh_l, self.kvh_l, self.hd, self.scale,
                        softcap=self.attn_softcap, window=window or 0,
                        split=self._ranges(B), kS=self.k_scale[i],
                        vS=self.v_scale[i], batch=B)
            if self.gemma:
                ho.gemv_fp8_mx(lw["wo_q"], lw["wo_s"], self.b_att, t1, B,
                               nhh, H)
                ho.gemv_fp8_mx(lw["wgu_q"], lw["wgu_s"], t1, gu, B, H,
                               2 * I, stage=ho.STAGE_NORM2, x2=h,
                               x2stride=H, g=lw["g_post"],
                               g2=lw["g_preffn"], hout=hb, hstride=H,
                               eps=eps)
                h, hb = hb, h
                ho.gemv_fp8_mx(lw["wdown_q"], lw["wdown_s"], gu, t2, B,
                               2 * I, H, stage=ho.STAGE_GLU,
                               x2=gu[:, I:], x2stride=2 * I, act=self.act)
            else:
                ho.gemv_fp8_mx(lw["wo_q"], lw["wo_s"], self.b_att, h, B,
                               nhh, H, res=h, rstride=H)
                ho.gemv_fp8_mx(lw["wgu_q"], lw["wgu_s"], h, gu, B, H,
                               2 * I, stage=ho.STAGE_NORM, g=lw["g_post"],
                               eps=eps)
                ho.gemv_fp8_mx(lw["wdown_q"], lw["wdown_s"], gu, h, B,
                               2 * I, H, stage=ho.STAGE_GLU, x2=gu[:, I:],
                               x2stride=2 * I, act=self.act, res=h,
                               rstride=H)
        if self.gemma:
            ho.gemv_fp8_mx(self.lm_head_q, self.lm_head_s, t2,
                           self.bt_logits, B, H, self.vocab_l,
                           stage=ho.STAGE_NORM2, x2=h, x2stride=H,
                           g=self.layers[-1]["g_postffn"], g2=self.g_final,
                           hout=hb, hstride=H, eps=eps,
                           softcap=self.final_softcap)
        else:
            ho.gemv_fp8_mx(self.lm_head_q, self.lm_head_s, h,
                           self.bt_logits, B, H, self.vocab_l,
                           stage=ho.STAGE_NORM, g=self.g_final, eps=eps,
                           softcap=self.final_softcap)
        ho.sample(self.bt_logits[:B], min_p, greedy, self.seed,
                  self.rng_ctr, self.bt_gmax, self.bt_pick, self.bt_next,
                  self.bt_ring, self.bt_nout, self.bt_lens, bump_len=True,
                  temperature=temperature, cnt=self.bt_cnt, batch=B)

    def prefill_batch(self, prompts) -> None:
        """Prefill B prompts (RAGGED lengths allowed) into per-sequence
        KV pools; each row then decodes from its own position
        (bt_lens[b] device-side)."""
        seqs = [np.asarray(p, dtype=np.int32).ravel() for p in prompts]
        B = len(seqs)
        assert 1 <= B <= self.max_batch and self.max_batch > 1
        assert self.world == 1, "batched decode is single-GPU for now"
        lens = [len(sq) for sq in seqs]
        if min(lens) == 0:
            raise ValueError("empty prompt in batch")
        if max(lens) + 1 >= self.max_seq:
            raise ValueError(f"prompt {max(lens)} fills the "
                             f"{self.max_seq} pool")
        self.reset()
        self.bt_nout.zero_()
        for segs in self._chunks(lens, self._chunk_rows):
            if len(segs) > 1:
                self._read_pack(segs, seqs)
                continue
            (b, done, M), = segs
            self._pb = b
            self._read(seqs[b][done:done + M], done)
            if done + M == lens[b]:
                self._heads([(b, M - 1)], B)
        self._pb = 0
        self.bt_lens[:B].copy_(torch.tensor(lens, dtype=torch.int32))
        self._host_lens = lens
        self._batch_n = B

    def _chunks(self, lens, rows=None):
        """The prompts in chunks of up to PC rows, each a list of (sequence,
        first position, rows); a prompt whose chunks are its own in chunks of
        rows(its length), as it is read elsewhere.  Several prompts share a
        chunk, so that its
        products have the rows of all: read one by one, 16 prompts of 305 to
        611 rows beside e4m3 weights left tiles half empty and W was streamed
        16 times (with 31 steps behind them 17.5 -> 13.4 ms; six of 167 to
        333 in bf16 with 23 steps 10.1 -> 8.4; prompts alone beside MXFP4,
        eight layers of 3584: 16 of 305 to 611 rows 74 ms one by one in
        products of their own, 27 so).  Beside e4m3 weights a row in a chunk
        by itself is not rounded to e4m3, so which rows are must not depend on
        a prompt's neighbours: the ones that end with such a row go alone, and
        of the others none is left with one (the cut before it moves up)."""
        e4m3 = self.fp8 and not self.wq4
        apart = self.hd not in (64, 128, 256) or (e4m3 and self.PC < 3)
        chunks, room = [], 0
        for b, n in enumerate(lens):
            alone = apart or (e4m3 and n % self.PC == 1)
            own = rows and (alone or len(lens) == 1)
            most = rows(n) if own else self.PC
            done = 0
            while done < n:
                if alone or room == 0:
                    chunks.append([])
                    room = most
                M = min(n - done, room)
                if e4m3 and not alone and n - done - M == 1:
                    M, room = M - 1, M - 1
                if M:
                    chunks[-1].append((b, done, M))
                done += M
                room = 0 if alone else room - M
        return chunks

    def _read_pack(self, segs, seqs) -> None:
        """One chunk of several prompts through the layers, and the logits of
        those that it ends."""
        M = sum(n for _, _, n in segs)
        ends, row = [], 0
        for b, done, n in segs:
            row += n
            if done + n == len(seqs[b]):
                ends.append((b, row - 1))
        tiles = ho.attn_tiles(segs, self.nh_l // self.kvh_l)
        parts = [np.concatenate([seqs[b][p:p + n] for b, p, n in segs]),
                 np.concatenate([np.arange(p, p + n) for _, p, n in segs]),
                 np.repeat([b for b, _, _ in segs], [n for _, _, n in segs]),
                 tiles.ravel(), np.array([r for _, r in ends])]
        host = np.concatenate(parts).astype(np.int32)
        buf = self.pack_buf[:len(host)]
        buf.copy_(torch.from_numpy(host))
        ids, rows, tiles, last = buf.split(
            [M, 2 * M, tiles.size, len(ends)])
        self._stack.embed(ids, M, 0)
        self._layers_forward(
            M, keys=max(p + n for _, p, n in segs),
            pack=(rows, tiles.view(-1, 5), max(n for _, _, n in segs)))
        self._heads(ends, len(seqs), last)

    def _heads(self, ends, B: int, last=None) -> None:
        """The logits of sequences b whose last row is r, `ends` of them (b,
        r), of a group of B; last: the r, int32 on the device."""
        if self.wq4 or self.tp_branch or B == 1 or (
                self.H % 64 if self.fp8 else len(ends) == 1):
            for b, r in ends:
                self._lm_head_last(r + 1)
                self.bt_logits32[b].copy_(self.b_logits)
            return
        if self.fp8:
            # Not rounded to e4m3, W read once for 16.  By itself a row's sums
            # would go in another order, so a single one of a group goes here
            # too (40 us instead of 22, 32768x3584): its logits do not depend
            # on which prompts end beside it.  A prompt without a group has
            # the product of one row.
            x = self.b_h
            if last is None:
                (_, r), = ends
                x, last = x[r:r + 1], self.b_row0
            for i in range(0, len(ends), ho.HEAD_ROWS):
                n = min(len(ends) - i, ho.HEAD_ROWS)
                b = ends[i][0]
                ho.head_rows(x, last[i:], self.lm_head_q, self.lm_head_s,
                             self.bt_logits32[b:b + n], n, self.g_final,
                             self.b_parts, eps=self.config.rms_norm_eps,
                             softcap=self.final_softcap)
            return
        # bf16: a row is the same among others, W is read once for 16
        for i in range(0, len(ends), ho.FEW_ROWS):
            n = min(len(ends) - i, ho.FEW_ROWS)
            b = ends[i][0]
            ho.embed(self.b_h, last[i:], self.b_t1, n)
            self._rows(self._head, "", self.b_t1, self.bt_logits32[b:b + n],
                       n, g=self.g_final, softcap=self.final_softcap)

    # ---- continuous batching primitives (rows join/leave the group) ----
    def prefill_row(self, b: int, ids, greedy: bool = True,
                    min_p: float = 0.1, temperature: float = 1.0):
        """Prefill ONE sequence into slot b (other rows untouched) and
        sample its first token — a request JOINING the lockstep group
        between decode chunks (server continuous batching)."""
        ids = np.asarray(ids, dtype=np.int32).ravel()
        P = len(ids)
        if P == 0:
            raise ValueError("empty prompt")
        assert 0 <= b < self.max_batch and self.max_batch > 1
        assert self.world == 1
        if P + 1 >= self.max_seq:
            raise ValueError(f"prompt {P} fills the {self.max_seq} pool")
        self._pb = b
        done = 0
        rows = self._chunk_rows(P)
        while done < P:
            M = min(P - done, rows)
            self._read(ids[done:done + M], done)
            done += M
        self._lm_head_last(M)
        self._pb = 0
        self.bt_lens[b:b + 1].fill_(P)
        self.bt_nout[b:b + 1].zero_()
        # first token for this row only (row-sliced sampler state)
        ho.sample(self.b_logits, min_p, greedy, self.seed, self.rng_ctr,
                  self.bt_gmax[b:b + 1], self.bt_pick[b:b + 1],
                  self.bt_next[b:b + 1], self.bt_ring[b:b + 1],
                  self.bt_nout[b:b + 1], self.bt_lens[b:b + 1],
                  bump_len=False, temperature=temperature,
                  cnt=self.bt_cnt[b:b + 1], batch=1)
        if not hasattr(self, "_host_lens") or self._host_lens is None:
            self._host_lens = [0] * self.max_batch
        while len(self._host_lens) < self.max_batch:
            self._host_lens.append(0)
        self._host_lens[b] = P
        self._batch_n = max(getattr(self, "_batch_n", 0), b + 1)

    def compact_row(self, dst: int, src: int):
        """Move sequence slot src -> dst (KV pools, scales, device row
        state) so retired rows leave the group dense."""
        if dst == src:
            return
        for i in range(self.config.num_hidden_layers):
            self.k_cache[i][dst].copy_(self.k_cache[i][src])
            self.v_cache[i][dst].copy_(self.v_cache[i][src])
            if self.kv8:
                self.k_scale[i][dst].copy_(self.k_scale[i][src])
                self.v_scale[i][dst].copy_(self.v_scale[i][src])
        for t in (self.bt_lens, self.bt_next, self.bt_nout, self.bt_gmax,
                  self.bt_pick, self.bt_cnt):
            t[dst:dst + 1].copy_(t[src:src + 1])
        self.bt_ring[dst].copy_(self.bt_ring[src])
        self._host_lens[dst] = self._host_lens[src]
