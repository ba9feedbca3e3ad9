"""ctypes bindings for the hand-written CDNA4 kernel library.

The library (``_libllmops.so``, built in-tree by ``csrc/build.py`` /
``__graft_entry__.build()``) exposes plain-C launch functions taking raw
device pointers + the HIP stream; tensors stay ``torch`` tensors (memory
containers only) and every launch lands on the *current* torch stream, so
the whole decode step can be captured in a hipGraph via
``torch.cuda.CUDAGraph``.

This module fails loudly if the extension is missing while a GPU is
present — there is no silent eager fallback (the HIP path must be the one
that runs).
"""

from __future__ import annotations

import ctypes
import os

import numpy as np
import torch

from . import tape as _tape

_LIB = None
_LIB_PATH = os.path.join(os.path.dirname(os.path.dirname(
    os.path.abspath(__file__))), "_libllmops.so")

_SIGS = {
    "launch_gemv": [ctypes.c_void_p] * 9 + [ctypes.c_int] * 8 +
                   [ctypes.c_float] * 3 +
                   [ctypes.c_int, ctypes.c_void_p, ctypes.c_int] +
                   [ctypes.c_long] * 2 + [ctypes.c_void_p] * 2 +
                   [ctypes.c_long, ctypes.c_void_p],
    "launch_rmsnorm": [ctypes.c_void_p] * 8 + [ctypes.c_int] * 2 +
                      [ctypes.c_float, ctypes.c_void_p],
    "launch_rope_cache": [ctypes.c_void_p] * 7 + [ctypes.c_int] +
                         [ctypes.c_void_p] * 4 + [ctypes.c_int] * 7 +
                         [ctypes.c_void_p],
    "launch_attn": [ctypes.c_void_p] * 7 + [ctypes.c_int] * 7 +
                   [ctypes.c_float, ctypes.c_float, ctypes.c_int,
                    ctypes.c_void_p],
    "launch_attn_prefill_mfma": [ctypes.c_void_p] * 9 + [ctypes.c_long] +
                                [ctypes.c_int] * 10 +
                                [ctypes.c_float, ctypes.c_float,
                                 ctypes.c_int, ctypes.c_void_p],
    "launch_attn_dec": [ctypes.c_void_p] * 9 + [ctypes.c_int] +
                       [ctypes.c_void_p] * 2 + [ctypes.c_int] * 6 +
                       [ctypes.c_float, ctypes.c_float, ctypes.c_int,
                        ctypes.c_void_p],
    "launch_glu": [ctypes.c_void_p] * 3 + [ctypes.c_long, ctypes.c_int,
                                           ctypes.c_void_p],
    "launch_embed": [ctypes.c_void_p] * 3 + [ctypes.c_int] * 2 +
                    [ctypes.c_float, ctypes.c_void_p],
    "launch_sample": [ctypes.c_void_p, ctypes.c_int, ctypes.c_int,
                      ctypes.c_int, ctypes.c_long, ctypes.c_float,
                      ctypes.c_int, ctypes.c_uint64, ctypes.c_float] +
                     [ctypes.c_void_p] * 8 +
                     [ctypes.c_int, ctypes.c_void_p, ctypes.c_int,
                      ctypes.c_void_p],
    "launch_gemm_prompt": [ctypes.c_void_p] * 9 + [ctypes.c_long] +
                          [ctypes.c_int] * 5 + [ctypes.c_void_p],
    "gemm_prompt_plan": [ctypes.c_int] * 5 + [ctypes.c_long, ctypes.c_int,
                                              ctypes.c_void_p],
    "launch_row_gemm": [ctypes.c_void_p] * 11 + [ctypes.c_long] +
                       [ctypes.c_int] * 11 +
                       [ctypes.c_float, ctypes.c_float, ctypes.c_void_p],
    "launch_mid_gemm": [ctypes.c_void_p] * 9 + [ctypes.c_long] +
                       [ctypes.c_int] * 9 + [ctypes.c_float, ctypes.c_void_p],
    "attn_prefill_plan": [ctypes.c_int] * 9 + [ctypes.c_long,
                                               ctypes.c_void_p],
    "row_gemm_plan": [ctypes.c_int] * 6 + [ctypes.c_long, ctypes.c_int,
                                           ctypes.c_void_p],
    "launch_prefetch": [ctypes.c_void_p, ctypes.c_long, ctypes.c_void_p,
                        ctypes.c_void_p],
    "launch_softcap": [ctypes.c_void_p, ctypes.c_long, ctypes.c_float,
                       ctypes.c_void_p],
    "launch_addinto": [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long,
                       ctypes.c_void_p],
    "launch_i32_set": [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p],
    "launch_quant_fp8": [ctypes.c_void_p] * 3 + [ctypes.c_int] * 3 +
                        [ctypes.c_void_p],
    "launch_quant_fp4": [ctypes.c_void_p] * 3 + [ctypes.c_int] * 2 +
                        [ctypes.c_void_p],
    "launch_head_rows": [ctypes.c_void_p] * 7 + [ctypes.c_int] * 3 +
                        [ctypes.c_float] * 2 + [ctypes.c_void_p],
    "launch_gemv_fp8_mx": [ctypes.c_void_p] * 3 + [ctypes.c_long] +
                          [ctypes.c_void_p, ctypes.c_long] +
                          [ctypes.c_void_p] * 3 + [ctypes.c_long] +
                          [ctypes.c_void_p, ctypes.c_long] +
                          [ctypes.c_void_p, ctypes.c_long] +
                          [ctypes.c_int] * 5 +
                          [ctypes.c_float, ctypes.c_int, ctypes.c_float,
                           ctypes.c_float, ctypes.c_void_p],
    "launch_gemm_fp4w": [ctypes.c_void_p] * 8 + [ctypes.c_long] +
                        [ctypes.c_int] * 5 + [ctypes.c_void_p],
    "launch_moe_route": [ctypes.c_void_p] * 3 + [ctypes.c_int] * 4 +
                        [ctypes.c_float] + [ctypes.c_void_p] * 4,
    "launch_expert_sort": [ctypes.c_void_p] * 2 + [ctypes.c_int] * 2 +
                          [ctypes.c_long, ctypes.c_void_p],
    "launch_expert_gemm": [ctypes.c_void_p] * 6 + [ctypes.c_int] * 7 +
                          [ctypes.c_void_p],
    "expert_gemm_plan": [ctypes.c_int] * 6 + [ctypes.c_void_p],
    "launch_expert_sum": [ctypes.c_void_p] * 4 + [ctypes.c_int] * 3 +
                         [ctypes.c_void_p],
    "launch_moe_scale_add": [ctypes.c_void_p] * 3 +
                            [ctypes.c_long, ctypes.c_int, ctypes.c_int,
                             ctypes.c_void_p],
    "stack_forward": [ctypes.c_void_p] + [ctypes.c_int] * 5 +
                     [ctypes.c_void_p] * 2 + [ctypes.c_int] * 2 +
                     [ctypes.c_void_p],
    "stack_chunk_rows": [ctypes.c_void_p, ctypes.c_int, ctypes.c_int],
    "stack_embed": [ctypes.c_void_p] * 3 + [ctypes.c_int] * 2 +
                   [ctypes.c_void_p],
    "chain_slots": [ctypes.c_void_p] + [ctypes.c_int] * 2,
    "launch_chain": [ctypes.c_void_p] + [ctypes.c_int] * 3 +
                    [ctypes.c_float, ctypes.c_int] + [ctypes.c_void_p] * 2,
    "tape_run": [ctypes.c_void_p] + [ctypes.c_int] * 2 +
                [ctypes.c_void_p] * 2,
    # one-shot xGMI collectives (csrc/xgmi_comm.hip)
    "launch_xgmi_coll": [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                         ctypes.c_int, ctypes.c_int, ctypes.c_long,
                         ctypes.c_long, ctypes.c_int, ctypes.c_int,
                         ctypes.c_long, ctypes.c_void_p],
    "xc_alloc": [ctypes.c_long, ctypes.c_void_p],
    "xc_free": [ctypes.c_void_p],
    "xc_memset": [ctypes.c_void_p, ctypes.c_int, ctypes.c_long],
    "xc_h2d": [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long],
    "xc_d2h": [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long],
    "xc_ipc_handle": [ctypes.c_void_p, ctypes.c_void_p],
    "xc_ipc_open": [ctypes.c_void_p, ctypes.c_void_p],
    "xc_ipc_close": [ctypes.c_void_p],
}


def lib():
    global _LIB
    if _LIB is None:
        if not os.path.exists(_LIB_PATH):
            raise RuntimeError(
                f"HIP kernel library not built: {_LIB_PATH} missing. "
                f"Run `python csrc/build.py` (or __graft_entry__.build()).")
        _LIB = ctypes.CDLL(_LIB_PATH)
        for name, argtypes in _SIGS.items():
            fn = getattr(_LIB, name)
            fn.argtypes = argtypes
            fn.restype = ctypes.c_int  # hipError_t
    return _tape.library(_LIB)


def record(step):
    """Runs step() and keeps its launches (see ops/tape.py)."""
    return _tape.record(step, lib())


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _check(err: int, name: str):
    if err != 0:
        raise RuntimeError(f"{name} failed: hipError_t={err}")


def _ptr(t) -> int:
    return 0 if t is None else t.data_ptr()


def _ld(t, width: int) -> int:
    """Elements from row to row: rows of one buffer may lie in another's;
    what is in one piece may have any shape."""
    return width if t.is_contiguous() else t.stride(0)


# ----------------------------------------------------------------------
# op wrappers (shapes validated here; kernels trust their args)
# ----------------------------------------------------------------------

STAGE_RAW, STAGE_NORM, STAGE_GLU, STAGE_NORM2 = 0, 1, 2, 3
# NORM_EMBED: W-input x is the embedding TABLE; the row at *x2 (device
# token id) is gathered, scaled by `escale` and normed — fuses the
# decode step's k_embed launch into the first QKV GEMV.  `res` receives
# the persisted h (residual stream).
STAGE_NORM_EMBED = 4


def _gemv(wt, W, ws, we, K, x, y, res, softcap, stage, x2, g, act, eps,
          maxblocks, g2, escale, eidx, wstride, sstride, oscale, glu,
          ones=None):
    N, ne = W.shape[0] // (2 if glu else 1), 1
    if eidx is not None:        # experts that there are rows for
        ne = min(eidx.numel(), y.numel() // N if glu else x.numel() // K)
        assert oscale is None or oscale.numel() >= ne
    _check(lib().launch_gemv(
        _ptr(W), _ptr(ws), _ptr(we), _ptr(x), _ptr(x2), _ptr(g), _ptr(g2),
        _ptr(y), _ptr(res), wt, N, K, stage, act, int(glu),
        int(x.dtype == torch.float32),
        int(y.dtype == torch.float32), ctypes.c_float(eps),
        ctypes.c_float(softcap), ctypes.c_float(escale), maxblocks,
        _ptr(eidx), ne, ctypes.c_long(wstride), ctypes.c_long(sstride),
        _ptr(oscale), _ptr(ones) or None,
        0 if ones is None else ones.numel() * ones.itemsize, _stream()),
        "gemv")


def gemv(W: torch.Tensor, x: torch.Tensor, y: torch.Tensor,
         res: torch.Tensor | None = None, softcap: float = 0.0,
         stage: int = 0, x2: torch.Tensor | None = None,
         g: torch.Tensor | None = None, act: int = 0, eps: float = 1e-5,
         nt: int = 1, rpw: int = 1, maxblocks: int = 0,
         g2: torch.Tensor | None = None, escale: float = 1.0,
         eidx: torch.Tensor | None = None, wstride: int = 0,
         oscale: torch.Tensor | None = None, glu: bool = False,
             ones: torch.Tensor | None = None):
    """y[N] = W[N,K] @ stage(x)[K] (+res); stage takes RMSNorm / GLU /
    the Gemma sandwich (NORM2: x2 = h_in, g/g2 = post/pre gammas, res =
    h_out ping-pong) / the embed gather (NORM_EMBED: x = embed table,
    x2 = token-id i32, res = persisted h) on the way.  x is bf16, or fp32
    (RAW).  glu: W holds gate rows, then up rows: y[N/2] = act(gate) * up.
    eidx/wstride/oscale: W of expert *eidx, its result times *oscale; of
    several experts (x [n, K]) the results are added up, with glu they stand
    one after the other (y [n, N/2]).  ones: a buffer filled with ones besides
    (``Chain``).  nt and rpw are kept for callers: the kernel streams
    W past the caches and picks its rows by itself."""
    _gemv(0, W, None, None, W.shape[1], x, y, res, softcap, stage, x2, g,
          act, eps, maxblocks, g2, escale, eidx, wstride, 0, oscale, glu, ones)


def gemv_fp8(Wq: torch.Tensor, scales: torch.Tensor, x: torch.Tensor,
             y: torch.Tensor, res: torch.Tensor | None = None,
             softcap: float = 0.0, stage: int = 0,
             x2: torch.Tensor | None = None, g: torch.Tensor | None = None,
             act: int = 0, eps: float = 1e-5, nt: int = 1, rpw: int = 1,
             maxblocks: int = 0, g2: torch.Tensor | None = None,
             escale: float = 1.0, eidx: torch.Tensor | None = None,
             wstride: int = 0, sstride: int = 0,
             oscale: torch.Tensor | None = None, glu: bool = False,
             ones: torch.Tensor | None = None):
    """y[N] = scales * (Wq[N,K] @ stage(x)); Wq = e4m3fn bytes; the rest
    as for gemv (sstride: scales of an expert)."""
    _gemv(1, Wq, scales, None, Wq.shape[1], x, y, res, softcap, stage, x2, g,
          act, eps, maxblocks, g2, escale, eidx, wstride, sstride, oscale,
          glu, ones)


def rmsnorm(x: torch.Tensor, g: torch.Tensor, y: torch.Tensor | None,
            res: torch.Tensor | None = None, eps: float = 1e-5,
            g2: torch.Tensor | None = None, y2: torch.Tensor | None = None,
            q2: torch.Tensor | None = None, s2: torch.Tensor | None = None):
    """y = norm(x)*g ; with res: y = res + norm(x)*g (Gemma post).  With g2
    also y2 = norm(y)*g2, the norm behind the residual, or the same as e4m3
    rows q2 with scales s2.  y None: norm(x)*g itself as e4m3 rows, rounded
    once."""
    M = 1 if x.dim() == 1 else x.shape[0]
    H = x.shape[-1]
    _check(lib().launch_rmsnorm(
        _ptr(x), _ptr(g), _ptr(res), _ptr(y), _ptr(g2), _ptr(y2), _ptr(q2),
        _ptr(s2), M, H,
        ctypes.c_float(eps), _stream()), "rmsnorm")


def rope_cache(q: torch.Tensor, k_in: torch.Tensor, v_in: torch.Tensor,
               k_cache: torch.Tensor, v_cache: torch.Tensor,
               cos_t: torch.Tensor, sin_t: torch.Tensor,
               pos_ptr: torch.Tensor, M: int, nh: int, kvh: int, hd: int,
               kS: torch.Tensor | None = None,
               vS: torch.Tensor | None = None,
               rows: torch.Tensor | None = None):
    """kS/vS given => fp8 (e4m3) KV pool with per-(head,pos) scales.
    q, k_in, v_in: M rows, which may lie in one fused buffer (k_in and v_in
    equally far apart).  rows (int32 [2, M]): the position of each row and
    which pool of several it belongs to (caches [pools, kvh, S, hd])."""
    S = k_cache.shape[-2]
    assert rows is None or (rows.numel() == 2 * M and k_cache.dim() == 4)
    assert _ld(v_in, kvh * hd) == _ld(k_in, kvh * hd)
    _check(lib().launch_rope_cache(
        _ptr(q), _ptr(k_in), _ptr(v_in), _ptr(k_cache), _ptr(v_cache),
        _ptr(kS), _ptr(vS), 1 if kS is not None else 0,
        _ptr(cos_t), _ptr(sin_t), _ptr(pos_ptr), _ptr(rows), M, nh, kvh, hd,
        S, _ld(q, nh * hd), _ld(k_in, kvh * hd), _stream()), "rope_cache")


def attn(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor,
         out: torch.Tensor, len_ptr: torch.Tensor, M: int, nh: int,
         kvh: int, hd: int, scale: float, softcap: float = 0.0,
         window: int = 0, kS: torch.Tensor | None = None,
         vS: torch.Tensor | None = None):
    S = k_cache.shape[1]
    _check(lib().launch_attn(
        _ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(out), _ptr(len_ptr),
        _ptr(kS), _ptr(vS), 1 if kS is not None else 0,
        M, nh, kvh, hd, _ld(q, nh * hd), S, ctypes.c_float(scale),
        ctypes.c_float(softcap), window, _stream()), "attn")


def attn_prefill_mfma(q: torch.Tensor, k_cache: torch.Tensor,
                      v_cache: torch.Tensor, out: torch.Tensor,
                      len_ptr: torch.Tensor, M: int, nh: int, kvh: int,
                      hd: int, scale: float, softcap: float = 0.0,
                      window: int = 0, kS: torch.Tensor | None = None,
                      vS: torch.Tensor | None = None,
                      part: torch.Tensor | None = None, keys: int = 0,
                      tiles: torch.Tensor | None = None, most: int = 0):
    """Flash prefill attention (MFMA, online softmax); q already roped,
    caches already written for [0, pos0+M).  With part (fp32 scratch) few
    rows split their keys over more blocks; keys (pos0+M, as far as the
    host knows) sizes that split.  tiles (``attn_tiles``): rows of several
    sequences, the longest of ``most`` rows, caches [pools, kvh, S, hd]."""
    S = k_cache.shape[-2]
    assert tiles is None or (tiles.shape[-1] == 5 and tiles.is_contiguous()
                             and k_cache.dim() == 4)
    _check(lib().launch_attn_prefill_mfma(
        _ptr(q), _ptr(k_cache), _ptr(v_cache), _ptr(out), _ptr(len_ptr),
        _ptr(tiles), _ptr(kS), _ptr(vS), _ptr(part),
        ctypes.c_long(0 if part is None else part.numel()),
        1 if kS is not None else 0,
        M, nh, kvh, hd, _ld(q, nh * hd), S, max(keys, M if not most else 1),
        most, 0 if tiles is None else tiles.shape[0], ctypes.c_float(scale),
        ctypes.c_float(softcap), window, _stream()), "attn_prefill_mfma")


def attn_prefill_plan(M: int, nh: int, kvh: int, hd: int, keys: int,
                      window: int = 0, kv8: bool = False, part: int = 1 << 62,
                      most: int = 0, ntiles: int = 0) -> dict:
    """How attn_prefill_mfma goes about a call with so many floats of part:
    ranges of keys, whether two groups of waves share a block's (two), whether
    parts of the ranges lie row by row (by_row).  Host arithmetic only."""
    out = (ctypes.c_int * 3)()
    _check(lib().attn_prefill_plan(
        int(kv8), M, nh, kvh, hd, max(keys, M if not most else 1), most,
        ntiles, window, ctypes.c_long(part),
        ctypes.cast(out, ctypes.c_void_p)), "attn_prefill_plan")
    return dict(ranges=out[0], two=bool(out[1]), by_row=bool(out[2]))


def attn_tiles(segs, group: int) -> np.ndarray:
    """The tiles of attn_prefill_mfma for segs [(pool, position, rows)],
    which follow each other in the batch, ``group`` query heads to a kv head:
    those that see the most keys first."""
    per = 32 if max(n for _, _, n in segs) * group <= 32 else 128
    out, row0 = [], 0
    for pool, pos, n in segs:
        t = np.arange(-(-n * group // per))
        last = pos + np.minimum(n, -(-(t + 1) * per // group))   # keys seen
        out.append(np.stack([t, np.full_like(t, row0), np.full_like(t, n),
                             np.full_like(t, pos), np.full_like(t, pool),
                             last]))
        row0 += n
    t = np.concatenate(out, axis=1)
    return t[:5, np.argsort(-t[5], kind="stable")].T.astype(np.int32)


def attn_dec(qkv: torch.Tensor, k_cache: torch.Tensor,
             v_cache: torch.Tensor, out: torch.Tensor,
             len_ptr: torch.Tensor, cos_t: torch.Tensor,
             sin_t: torch.Tensor, scratch: torch.Tensor,
             cnt: torch.Tensor, nh: int, kvh: int, hd: int,
             scale: float, softcap: float = 0.0, window: int = 0,
             split: int = 1, kS: torch.Tensor | None = None,
             vS: torch.Tensor | None = None, batch: int = 1):
    """Fused decode attention: RoPE(q,k) + KV write + online softmax, the
    history in up to `split` ranges (as many as the device finds worth it;
    last-arriver merge).  kS/vS given => fp8 KV pool (quantized write +
    dequant scan).  batch>1: lockstep sequence rows, each with its own
    position, KV pool, scratch and tickets."""
    S = k_cache.shape[-2]
    _check(lib().launch_attn_dec(
        _ptr(qkv), _ptr(k_cache), _ptr(v_cache), _ptr(out), _ptr(len_ptr),
        _ptr(cos_t), _ptr(sin_t), _ptr(kS), _ptr(vS),
        1 if kS is not None else 0,
        _ptr(scratch), _ptr(cnt), split, batch,
        nh, kvh, hd, S, ctypes.c_float(scale),
        ctypes.c_float(softcap), window, _stream()), "attn_dec")


def glu(gate: torch.Tensor, up: torch.Tensor, out: torch.Tensor, act: int):
    """out = act(gate) * up; act 0 = SiLU, 1 = tanh-GELU."""
    total = gate.numel()
    assert total % 8 == 0
    _check(lib().launch_glu(_ptr(gate), _ptr(up), _ptr(out), total, act,
                            _stream()), "glu")


def embed(table: torch.Tensor, ids: torch.Tensor, out: torch.Tensor,
          M: int, scale: float = 1.0):
    H = table.shape[1]
    _check(lib().launch_embed(_ptr(table), _ptr(ids), _ptr(out), M, H,
                              ctypes.c_float(scale), _stream()), "embed")


def sample(logits: torch.Tensor, min_p: float, greedy: bool, seed: int,
           ctr: torch.Tensor, gmax: torch.Tensor, pick: torch.Tensor,
           next_token: torch.Tensor, out_ring: torch.Tensor,
           nout: torch.Tensor, len_ptr: torch.Tensor,
           bump_len: bool = True, temperature: float = 1.0,
           cnt: torch.Tensor | None = None, batch: int = 1,
           tops: torch.Tensor | None = None):
    """min-p / greedy sampler: parallel max + Gumbel-argmax; the
    last-arriving pick block commits the winner (no 1-thread fin
    launch).  gmax/pick are u64 scratch (zeroed once; the commit path
    re-zeros); tops (fp32, one row): the largest of shares that make up all
    logits, where their producer left them; cnt is an i32 ticket counter (zeroed once, re-armed).
    Temperature scales device-side (min-p keep-set + Gumbel score), so
    the GPU fast path matches the CPU sample_token() semantics."""
    V = logits.shape[-1]
    lbf16 = 1 if logits.dtype == torch.bfloat16 else 0
    ring_stride = out_ring.shape[-1] if out_ring.dim() > 1 else 0
    if batch > 1:
        assert (gmax.numel() >= batch and pick.numel() >= batch
                and next_token.numel() >= batch and nout.numel() >= batch
                and cnt is not None and cnt.numel() >= batch)
    if cnt is None:
        global _SAMPLE_CNT
        try:
            _SAMPLE_CNT
        except NameError:
            _SAMPLE_CNT = {}
        key = logits.device
        if key not in _SAMPLE_CNT:
            _SAMPLE_CNT[key] = torch.zeros(1, dtype=torch.int32,
                                           device=logits.device)
        cnt = _SAMPLE_CNT[key]
    inv_temp = 1.0 / max(float(temperature), 1e-6)
    _check(lib().launch_sample(
        _ptr(logits), V, lbf16, batch, ctypes.c_long(ring_stride),
        ctypes.c_float(min_p), 1 if greedy else 0,
        ctypes.c_uint64(seed), ctypes.c_float(inv_temp),
        _ptr(ctr), _ptr(gmax), _ptr(pick), _ptr(cnt),
        _ptr(next_token), _ptr(out_ring), _ptr(nout), _ptr(len_ptr),
        1 if bump_len else 0, _ptr(tops),
        0 if tops is None else tops.numel(), _stream()), "sample")


def _gemm_prompt(name, x, w, sx, sw, y, M, K, res, bias, act, accbuf, cnt):
    N = w.shape[0] // (2 if act >= 0 else 1)
    assert w.shape[1] == K and K % 64 == 0
    _check(lib().launch_gemm_prompt(
        _ptr(x), _ptr(w), _ptr(sx), _ptr(sw), _ptr(res), _ptr(bias), _ptr(y),
        _ptr(accbuf), _ptr(cnt),
        ctypes.c_long(0 if accbuf is None else accbuf.numel()),
        0 if cnt is None else cnt.numel(), M, N, K, act, _stream()), name)


def gemm(X: torch.Tensor, W: torch.Tensor, Y: torch.Tensor,
         res: torch.Tensor | None = None,
         accbuf: torch.Tensor | None = None,
         bias: torch.Tensor | None = None, act: int = -1,
         cnt: torch.Tensor | None = None):
    """Y[M,N] = X[M,K] @ W[N,K]^T (+bias, +res), bf16, MFMA prefill path.
    act 0/1: W holds gate rows, then up rows, and Y = act(gate) * up.
    accbuf (fp32) and cnt (int32, zero; left zero) let K be split over
    blocks where there are few tiles."""
    M, K = X.shape
    _gemm_prompt("gemm", X, W, None, None, Y, M, K, res, bias, act, accbuf,
                 cnt)


def gemm_prompt_plan(kind: str, M: int, N: int, K: int, act: int = -1,
                     part: int = 1 << 62, cnt: int = 1024) -> dict | None:
    """How gemm ("bf16"), gemm_fp8 and gemm_fp4w go about a product with so
    many floats of accbuf and counters: rows and outputs of a tile, parts of K,
    whether by the two groups of waves that take turns (wide), whether W is read
    past the caches (once), waves of a block; None: by mid_gemm.  Host arithmetic
    only."""
    out = (ctypes.c_int * 6)()
    _check(lib().gemm_prompt_plan(
        ("bf16", "fp8", "fp4").index(kind), M, N, K, act, ctypes.c_long(part),
        cnt, ctypes.cast(out, ctypes.c_void_p)), "gemm_prompt_plan")
    if not out[0]:
        return None
    return dict(rows=out[0], outputs=out[1], parts=out[2], wide=bool(out[3]),
                once=bool(out[4]), waves=out[5])


FEW_ROWS = 16        # rows that row_gemm takes
ROW_NORM_K = 4096    # the longest row that it norms


def row_gemm(x: torch.Tensor, w: torch.Tensor, y: torch.Tensor, M: int,
             ws: torch.Tensor | None = None,
             we: torch.Tensor | None = None,
             g: torch.Tensor | None = None, eps: float = 1e-5,
             bias: torch.Tensor | None = None,
             res: torch.Tensor | None = None, act: int = -1,
             softcap: float = 0.0, part: torch.Tensor | None = None,
             cnt: torch.Tensor | None = None,
             sx: torch.Tensor | None = None, norm16: bool = False):
    """Y[M<=16, N] = X W^T for few rows of x (2-D, rows may be apart), W
    streamed once: bf16, e4m3 (ws: row scales) or MXFP4 (we: exponents).
    x is bf16; beside e4m3 weights its rows are rounded to e4m3: by the
    caller (x bytes, sx scales), or after the norm that is taken here.
    g: RMSNorm of x on the way (K <= ROW_NORM_K; norm16: rounded to bf16
    before e4m3).  act 0/1: w holds gate
    rows, then up rows, and Y = act(gate) * up.  Then softcap, bias, res.
    part (fp32) and cnt (int32, zero; left zero) let K be split; where long
    rows need that and part is too small, fewer rows go at a time."""
    wt = 1 if ws is not None else 2 if we is not None else 0
    K = x.shape[-1]
    N = w.shape[0] // (2 if act >= 0 else 1)
    assert w.shape[1] * (2 if wt == 2 else 1) == K and w.is_contiguous()
    assert x.stride(-1) == 1 and y.stride(-1) == 1
    assert x.dtype == (torch.uint8 if wt == 1 and g is None
                       else torch.bfloat16)
    _check(lib().launch_row_gemm(
        _ptr(x), _ptr(sx), _ptr(w), _ptr(ws), _ptr(we), _ptr(g), _ptr(bias),
        _ptr(res), _ptr(y), _ptr(part), _ptr(cnt),
        ctypes.c_long(0 if part is None else part.numel()),
        0 if cnt is None else cnt.numel(), wt, M, N, K, x.stride(0),
        res.stride(0) if res is not None else 0, y.stride(0), act,
        1 if y.dtype == torch.float32 else 0, int(norm16),
        ctypes.c_float(eps), ctypes.c_float(softcap), _stream()), "row_gemm")


def mid_gemm(x: torch.Tensor, w: torch.Tensor, y: torch.Tensor, M: int,
             ws: torch.Tensor | None = None, sx: torch.Tensor | None = None,
             bias: torch.Tensor | None = None,
             res: torch.Tensor | None = None, act: int = -1,
             softcap: float = 0.0, part: torch.Tensor | None = None,
             cnt: torch.Tensor | None = None):
    """Y[M<=64, N] = X W^T, bf16 or e4m3 (x bytes, sx and ws scales of rows),
    the rest as for row_gemm without a norm (gate: up to 32 rows).  row_gemm
    and gemm hand on what it is faster for."""
    K, N = x.shape[-1], w.shape[0] // (2 if act >= 0 else 1)
    assert w.shape[1] == K and w.is_contiguous() and (sx is None) == \
        (ws is None)
    assert x.stride(-1) == 1 and y.stride(-1) == 1
    _check(lib().launch_mid_gemm(
        _ptr(x), _ptr(w), _ptr(sx), _ptr(ws), _ptr(res), _ptr(bias), _ptr(y),
        _ptr(part), _ptr(cnt),
        ctypes.c_long(0 if part is None else part.numel()),
        0 if cnt is None else cnt.numel(), M, N, K, x.stride(0),
        res.stride(0) if res is not None else 0, y.stride(0), act,
        1 if y.dtype == torch.float32 else 0, ctypes.c_float(softcap),
        _stream()), "mid_gemm")


def row_gemm_plan(kind: str, M: int, N: int, K: int, glu: bool = False,
                  norm: bool = False, part: int = 1 << 62,
                  cnt: int = 256) -> dict | None:
    """How row_gemm goes about a product with so many floats of part and
    counters (None: it does not take it).  Host arithmetic only."""
    out = (ctypes.c_long * 8)()
    if lib().row_gemm_plan(("bf16", "fp8", "fp4").index(kind), int(glu),
                           int(norm), M, N, K, ctypes.c_long(part), cnt,
                           ctypes.cast(out, ctypes.c_void_p)):
        return None
    return dict(zip(("rows", "splits", "k", "outputs", "tile", "blocks",
                     "lds", "floats"), out))


def row_gemm_room(kind: str, N: int, K: int, glu: bool = False) -> int:
    """Floats of part with which any number of rows goes in one launch."""
    plans = [row_gemm_plan(kind, M, N, K, glu) for M in range(1, FEW_ROWS + 1)]
    return max(p["floats"] if p else 0 for p in plans)


def quant_fp8(x: torch.Tensor, q: torch.Tensor, s: torch.Tensor):
    """Per-row e4m3fn quantization on device: q = fp8(x / s_row),
    s_row = absmax/448.  x: (M,K) bf16 or fp32, contiguous; q: >= M*K uint8;
    s: >= M fp32.  Used for weights at load and activations per GEMM."""
    M = 1 if x.dim() == 1 else x.shape[0]
    K = x.shape[-1]
    assert q.numel() >= M * K and s.numel() >= M
    _check(lib().launch_quant_fp8(_ptr(x), _ptr(q), _ptr(s),
                                  1 if x.dtype == torch.float32 else 0, M, K,
                                  _stream()), "quant_fp8")


def quant_fp4(x: torch.Tensor, q: torch.Tensor, e: torch.Tensor):
    """MXFP4 (OCP MX) weight quantization on device: e2m1 nibbles packed
    2/byte + one e8m0 scale byte per 32 elements.  x: (M,K) bf16;
    q: >= M*K/2 uint8; e: >= M*K/32 uint8."""
    M = 1 if x.dim() == 1 else x.shape[0]
    K = x.shape[-1]
    assert q.numel() >= M * K // 2 and e.numel() >= M * K // 32
    _check(lib().launch_quant_fp4(_ptr(x), _ptr(q), _ptr(e), M, K,
                                  _stream()), "quant_fp4")


def gemv_fp4(Wq: torch.Tensor, We: torch.Tensor, x: torch.Tensor,
             y: torch.Tensor, res: torch.Tensor | None = None,
             softcap: float = 0.0, stage: int = 0,
             x2: torch.Tensor | None = None, g: torch.Tensor | None = None,
             act: int = 0, eps: float = 1e-5, nt: int = 1, rpw: int = 1,
             maxblocks: int = 0, g2: torch.Tensor | None = None,
             escale: float = 1.0, glu: bool = False,
             ones: torch.Tensor | None = None):
    """y[N] = W4[N,K] @ stage(x): MXFP4 weights (Wq: N x K/2 packed
    bytes, We: N x K/32 e8m0 scale bytes) — half the fp8 stream; the rest
    as for gemv."""
    _gemv(2, Wq, None, We, Wq.shape[1] * 2, x, y, res, softcap, stage, x2, g,
          act, eps, maxblocks, g2, escale, None, 0, 0, None, glu, ones)


def gemm_fp8(xq: torch.Tensor, sx: torch.Tensor, Wq: torch.Tensor,
             sw: torch.Tensor, y: torch.Tensor, M: int, K: int,
             res: torch.Tensor | None = None,
             accbuf: torch.Tensor | None = None,
             bias: torch.Tensor | None = None, act: int = -1,
             cnt: torch.Tensor | None = None):
    """Y[M,N] = (sx_m * sw_n) * Xq[M,K] @ Wq[N,K]^T (+bias, +res): fp8 MFMA
    prefill path (both operands e4m3 with per-row scales); the rest as in
    gemm."""
    _gemm_prompt("gemm_fp8", xq, Wq, sx, sw, y, M, K, res, bias, act, accbuf,
                 cnt)


def gemv_fp8_mx(Wq: torch.Tensor, scales: torch.Tensor, x: torch.Tensor,
                y: torch.Tensor, B: int, xstride: int, ystride: int,
                res: torch.Tensor | None = None, rstride: int = 0,
                hout: torch.Tensor | None = None, hstride: int = 0,
                softcap: float = 0.0, stage: int = 0,
                x2: torch.Tensor | None = None, x2stride: int = 0,
                g: torch.Tensor | None = None,
                g2: torch.Tensor | None = None, act: int = 0,
                eps: float = 1e-5, escale: float = 1.0):
    """Multi-x fp8 GEMV: y[b, N] = scales * (Wq @ stage(x_b)) for B
    lockstep rows — one weight stream, B accumulators.  Strides are in
    ELEMENTS.  NORM_EMBED: x = embed table, x2 = int32 token ids."""
    N, K = Wq.shape
    out_f32 = 1 if y.dtype == torch.float32 else 0
    _check(lib().launch_gemv_fp8_mx(
        _ptr(Wq), _ptr(scales), _ptr(x), ctypes.c_long(xstride),
        _ptr(x2), ctypes.c_long(x2stride), _ptr(g), _ptr(g2),
        _ptr(y), ctypes.c_long(ystride), _ptr(res), ctypes.c_long(rstride),
        _ptr(hout), ctypes.c_long(hstride), N, K, B, stage, act,
        ctypes.c_float(eps), out_f32, ctypes.c_float(softcap),
        ctypes.c_float(escale), _stream()), "gemv_fp8_mx")


HEAD_ROWS = 16       # rows that head_rows takes


def head_rows(x: torch.Tensor, rows: torch.Tensor, Wq: torch.Tensor,
              scales: torch.Tensor, y: torch.Tensor, M: int, g: torch.Tensor,
              parts: torch.Tensor, eps: float = 1e-5, softcap: float = 0.0):
    """y[i] = softcap(norm(x[rows[i]]) Wq^T), M <= HEAD_ROWS rows beside e4m3
    weights that are not rounded to e4m3 themselves, W streamed once; y fp32.
    parts: scratch of 3 * HEAD_ROWS * K bf16."""
    N, K = Wq.shape
    assert x.is_contiguous() and x.shape[-1] == K and \
        x.dtype == parts.dtype == torch.bfloat16
    assert rows.dtype == torch.int32 and rows.numel() >= M
    assert y.dtype == torch.float32 and y.is_contiguous() and \
        y.numel() >= M * N and scales.numel() >= N
    assert parts.numel() >= 3 * HEAD_ROWS * K and g.numel() >= K
    _check(lib().launch_head_rows(
        _ptr(x), _ptr(rows), _ptr(g), _ptr(Wq), _ptr(scales), _ptr(parts),
        _ptr(y), M, N, K, ctypes.c_float(eps), ctypes.c_float(softcap),
        _stream()), "head_rows")


def gemm_fp4w(X: torch.Tensor, Wq4: torch.Tensor, We4: torch.Tensor,
              Y: torch.Tensor, res: torch.Tensor | None = None,
              accbuf: torch.Tensor | None = None,
              bias: torch.Tensor | None = None, act: int = -1,
              cnt: torch.Tensor | None = None):
    """Y[M,N] = X[M,K] @ dequant(W4)[N,K]^T (+bias, +res): bf16-MFMA prefill
    over MXFP4 weights (single-copy fp4 engines; activations unquantized
    -> more accurate than the fp8 prefill path).  act, accbuf and cnt as
    gemm's; accbuf alone brings counters of the call's own."""
    M, K = X.shape
    if accbuf is not None and cnt is None:
        cnt = torch.zeros(1024, dtype=torch.int32, device=X.device)
    N = Wq4.shape[0] // (2 if act >= 0 else 1)
    assert Wq4.shape[1] * 2 == K and K % 64 == 0
    _check(lib().launch_gemm_fp4w(
        _ptr(X), _ptr(Wq4), _ptr(We4), _ptr(res), _ptr(bias), _ptr(Y),
        _ptr(accbuf), _ptr(cnt),
        ctypes.c_long(0 if accbuf is None else accbuf.numel()),
        0 if cnt is None else cnt.numel(), M, N, K, act, _stream()),
        "gemm_fp4w")


def prefetch(t: torch.Tensor, sink: torch.Tensor):
    """Stream t through the cache hierarchy (side-stream warmer)."""
    n = t.numel() * t.element_size() // 2  # treat as u16 elements
    _check(lib().launch_prefetch(_ptr(t), n, _ptr(sink), _stream()),
           "prefetch")


def softcap(y: torch.Tensor, cap: float):
    """in-place y = cap * tanh(y / cap) (bf16)."""
    total = y.numel()
    assert total % 8 == 0
    _check(lib().launch_softcap(_ptr(y), total, ctypes.c_float(cap),
                                _stream()), "softcap")


def addinto(y: torch.Tensor, a: torch.Tensor):
    """y += a (bf16)."""
    total = y.numel()
    assert total % 8 == 0
    _check(lib().launch_addinto(_ptr(y), _ptr(a), total, _stream()), "addinto")


def i32_set(buf: torch.Tensor, v: int):
    _check(lib().launch_i32_set(_ptr(buf), v, _stream()), "i32_set")


# ----------------------------------------------------------------------
# a prompt's rows through all layers in one call (csrc/stack.hip)
# ----------------------------------------------------------------------

STACK_IDS = 128      # tokens that come with the embedding's launch


class _StackLin(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("w", "s", "e")]


class _StackLayer(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in (
        "g_in", "g_post", "g_preffn", "g_postffn", "bqkv", "wg")] + \
        [(n, _StackLin) for n in ("qkv", "o", "gu", "down")] + \
        [(n, ctypes.c_void_p) for n in ("kc", "vc", "kS", "vS")] + \
        [("window", ctypes.c_long)]


class _StackPlan(ctypes.Structure):
    _fields_ = [("layers", ctypes.POINTER(_StackLayer))] + \
        [(n, ctypes.c_void_p) for n in (
            "embed", "cos", "sin", "h", "xn", "t1", "qkv", "att", "gate",
            "acc", "row_cnt", "tile_cnt", "xq", "sx", "len", "moe_idx",
            "moe_w", "moe_order", "pairs", "aq", "sa")] + \
        [(n, ctypes.c_long) for n in ("acc_floats", "order_room")] + \
        [(n, ctypes.c_int) for n in (
            "nlayers", "H", "I", "nh", "kvh", "hd", "S", "wt", "kv8",
            "gemma", "act", "E", "topk", "nrow_cnt", "ntile_cnt", "mfma",
            "rows", "pools")] + \
        [(n, ctypes.c_float) for n in ("eps", "scale", "softcap", "escale")]


class Stack:
    """An engine's layers as the native launcher reads them.  ``layers``: of
    each layer its tensors by field (a linear's as (w, scales, exponents));
    ``fields``: the plan's, tensors or numbers.  Holds what it points to."""

    def __init__(self, layers, **fields):
        self._held = (layers, fields)

        def put(to, values):
            for n, v in values.items():
                if isinstance(v, tuple):
                    v = _StackLin(*[None if t is None else _ptr(t)
                                    for t in v])
                elif v is None or isinstance(v, torch.Tensor):
                    v = None if v is None else _ptr(v)
                setattr(to, n, v)

        self._layers = (_StackLayer * len(layers))()
        for to, l in zip(self._layers, layers):
            put(to, l)
        self._plan = _StackPlan(layers=self._layers, nlayers=len(layers))
        put(self._plan, fields)
        self._at = ctypes.addressof(self._plan)

    def embed(self, ids, M: int, pos0: int):
        """Rows of M tokens into h, and pos0 into len: ids on the host (int32
        numpy, up to STACK_IDS) or on the device."""
        host = isinstance(ids, np.ndarray)
        assert not host or (ids.dtype == np.int32 and len(ids) == M
                            and ids.flags.c_contiguous)
        assert host or ids.numel() >= M
        _check(lib().stack_embed(
            self._at, ids.ctypes.data if host else None,
            None if host else ids.data_ptr(), M, pos0, _stream()),
            "stack_embed")

    def chunk_rows(self, n: int, most: int) -> int:
        """Rows of the chunks that n rows of a prompt are best read in, at
        most ``most``."""
        return lib().stack_chunk_rows(self._at, n, most)

    def forward(self, M: int, keys: int, pool: int = 0, first: int = 0,
                last: int | None = None, rows=None, tiles=None, most: int = 0):
        """Rows [0, M) of h through layers [first, last); rows, tiles, most
        as for rope_cache and attn_prefill_mfma."""
        assert tiles is None or (rows.numel() == 2 * M and
                                 tiles.shape[-1] == 5)
        _check(lib().stack_forward(
            self._at, M, keys, pool, first,
            len(self._layers) if last is None else last, _ptr(rows),
            _ptr(tiles), 0 if tiles is None else tiles.shape[0], most,
            _stream()), "stack_forward")


# ----------------------------------------------------------------------
# the products between two attentions of one row (csrc/chain.hip)
# ----------------------------------------------------------------------

CHAIN_RAW, CHAIN_NORM, CHAIN_NORM2 = 0, 1, 2
# how long a wave waits for others' words before it looks for blocks that have
# not started, in steps of some 1.6 us.  ms for 200 tokens beside another
# stream's prompts and decode: 4 steps 537 and 270, 16 460 and 260, 32 414 and 360
CHAIN_LIMIT = 16
CHAIN_BLOCKS = 256
CHAIN_CLAIMS = CHAIN_BLOCKS * 4           # bytes of a launch's claims


def chain_room(n: int, dtype) -> int:
    """Bytes of n values that products of a chain leave each other."""
    return -(-n * dtype.itemsize // 256) * 256


def chain_part(buf: torch.Tensor, at: int, n: int, dtype) -> torch.Tensor:
    """n values at byte `at` of buf."""
    return buf[at:at + n * dtype.itemsize].view(dtype)


class _ChainStage(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in (
        "w", "ws", "we", "x", "h", "g", "g2", "add", "y", "hout")] + \
        [(n, ctypes.c_int) for n in (
            "N", "K", "kind", "x_f32", "wait", "glu", "y_f32", "own")] + \
        [("softcap", ctypes.c_float), ("slot", ctypes.c_int),
         ("route", ctypes.c_void_p), ("add2", ctypes.c_void_p),
         ("wstep", ctypes.c_long), ("sstep", ctypes.c_long)] + \
        [(n, ctypes.c_int) for n in ("scaled", "same", "experts", "top")] + \
        [("tops", ctypes.c_void_p)]


CHAIN_TOPS = CHAIN_BLOCKS * 4             # shares of the last product's outputs
CHAIN_TOP, CHAIN_EXPERTS = 2, 8           # routed experts of a row, of at most


class Chain:
    """Products that follow each other, in one launch.  ``stages``: of each,
    its weight ``W`` (w, scales, exponents), ``x`` (of an earlier one of them:
    its y), ``y`` and, where it has them, kind, g, g2, h, hout, add, glu,
    softcap, as csrc/chain.hip has them; of routed experts, W of all
    ``experts`` one below the other, ``slot`` from 1, ``route`` and ``top``
    with the first, scaled, add2; of the last, ``tops``: the largest of
    CHAIN_TOPS shares of y.  Every y but the last lies in memory that held
    ones, all bits of them, before the step (``ones`` of ``gemv``), and so
    does ``claims``, CHAIN_CLAIMS bytes by which waves take over the rows of
    blocks that find no CU.  Holds what it points to."""

    def __init__(self, stages, wt: int, act: int, eps: float, claims=None):
        self._held, self._claims = stages, claims
        assert claims is None or (claims.is_contiguous() and claims.numel() *
                                  claims.itemsize >= CHAIN_CLAIMS)
        self.wt, self.act, self.eps = wt, act, eps
        self._stages = (_ChainStage * len(stages))()
        f32 = torch.float32
        for i, (to, s) in enumerate(zip(self._stages, stages)):
            w, ws, we = s["W"]
            x, y, add = s["x"], s["y"], s.get("add")
            to.w, to.ws, to.we = w.data_ptr(), _ptr(ws) or None, \
                _ptr(we) or None
            rows, K = w.shape[0], w.shape[1] * (2 if wt == 2 else 1)
            to.slot = s.get("slot", 0)
            tops = s.get("tops")
            assert tops is None or (tops.dtype == f32 and
                                    tops.numel() >= CHAIN_TOPS)
            to.tops = _ptr(tops) or None
            if to.slot:
                rows //= s["experts"]
                to.wstep = rows * w.shape[1] * w.element_size()
                to.sstep, to.experts = rows, s["experts"]
                to.scaled = int(s.get("scaled", False))
                to.same = int(i > 0 and x is stages[i - 1]["x"])
                route, add2 = s.get("route"), s.get("add2")
                to.route, to.add2 = _ptr(route) or None, _ptr(add2) or None
                to.top = s.get("top", 0)
                assert route is None or (
                    route.dtype == torch.bfloat16 and route.is_contiguous()
                    and route.shape == (to.experts, K))
                assert add2 is None or (add2.dtype == f32 and
                                        add2.numel() >= rows)
            to.glu = int(s.get("glu", False))
            to.N, to.K = rows // (2 if to.glu else 1), K
            to.kind = s.get("kind", CHAIN_RAW)
            to.softcap = s.get("softcap", 0.0)
            to.x, to.y = x.data_ptr(), y.data_ptr()
            to.x_f32, to.y_f32 = int(x.dtype == f32), int(y.dtype == f32)
            to.wait = int(any(x is t["y"] for t in stages[:i]))
            to.own = int(add is not None and
                         any(add is t["y"] for t in stages[:i]))
            to.add = _ptr(add) or None
            assert w.is_contiguous() and x.is_contiguous() and \
                y.is_contiguous()
            assert x.numel() >= K and y.numel() >= to.N
            assert add is None or (add.dtype == torch.bfloat16 and
                                   add.numel() >= to.N)
            assert x.dtype in (f32, torch.bfloat16) and \
                y.dtype in (f32, torch.bfloat16)
            for n, dt in dict(h=torch.bfloat16, hout=torch.bfloat16, g=f32,
                              g2=f32).items():
                t = s.get(n)
                assert t is None or (t.dtype == dt and t.numel() >= K)
                setattr(to, n, _ptr(t) or None)

    def fits(self) -> bool:
        """Whether the sizes are ones that the kernel takes, and faster than
        a launch for each."""
        return lib().chain_slots(self._stages, len(self._stages),
                                 self.wt) >= 3

    def run(self, limit: int = CHAIN_LIMIT):
        _check(lib().launch_chain(
            self._stages, len(self._stages), self.wt, self.act,
            ctypes.c_float(self.eps), limit, _ptr(self._claims) or None,
            _stream()), "chain")


# ----------------------------------------------------------------------
# one-shot xGMI collectives (csrc/xgmi_comm.hip) — raw-pointer plumbing
# for the peer-mapped comm buffers (outside torch's caching allocator so
# the IPC base pointer is stable)
# ----------------------------------------------------------------------

XC_MODE_AR_BF16, XC_MODE_AR_F32, XC_MODE_GATHER = 0, 1, 2
XC_OFF_EPOCH, XC_OFF_TICKET, XC_OFF_ERR = 64, 72, 76
XC_OFF_DATA = 4096
XC_IPC_HANDLE_BYTES = 64


def xc_alloc(nbytes: int) -> int:
    p = ctypes.c_void_p(0)
    _check(lib().xc_alloc(ctypes.c_long(nbytes), ctypes.byref(p)), "xc_alloc")
    return p.value


def xc_free(ptr: int):
    _check(lib().xc_free(ctypes.c_void_p(ptr)), "xc_free")


def xc_memset(ptr: int, val: int, nbytes: int):
    _check(lib().xc_memset(ctypes.c_void_p(ptr), val,
                           ctypes.c_long(nbytes)), "xc_memset")


def xc_h2d(dst: int, data: bytes):
    buf = (ctypes.c_char * len(data)).from_buffer_copy(data)
    _check(lib().xc_h2d(ctypes.c_void_p(dst), buf,
                        ctypes.c_long(len(data))), "xc_h2d")


def xc_d2h(src: int, nbytes: int) -> bytes:
    buf = (ctypes.c_char * nbytes)()
    _check(lib().xc_d2h(buf, ctypes.c_void_p(src),
                        ctypes.c_long(nbytes)), "xc_d2h")
    return bytes(buf)


def xc_ipc_handle(ptr: int) -> bytes:
    h = (ctypes.c_char * XC_IPC_HANDLE_BYTES)()
    _check(lib().xc_ipc_handle(ctypes.c_void_p(ptr), h), "xc_ipc_handle")
    return bytes(h)


def xc_ipc_open(handle: bytes) -> int:
    assert len(handle) == XC_IPC_HANDLE_BYTES
    buf = (ctypes.c_char * XC_IPC_HANDLE_BYTES).from_buffer_copy(handle)
    p = ctypes.c_void_p(0)
    _check(lib().xc_ipc_open(buf, ctypes.byref(p)), "xc_ipc_open")
    return p.value


def xc_ipc_close(ptr: int):
    _check(lib().xc_ipc_close(ctypes.c_void_p(ptr)), "xc_ipc_close")


def xgmi_coll(dst_ptr: int, src_ptr: int, mybase: int, rank: int,
              world: int, nbytes: int, slot_bytes: int, mode: int,
              nstripes: int, spin_limit: int = 5_000_000):
    """One one-shot collective on the current torch stream (capturable)."""
    _check(lib().launch_xgmi_coll(
        ctypes.c_void_p(dst_ptr), ctypes.c_void_p(src_ptr),
        ctypes.c_void_p(mybase), rank, world, ctypes.c_long(nbytes),
        ctypes.c_long(slot_bytes), mode, nstripes,
        ctypes.c_long(spin_limit), _stream()), "xgmi_coll")


def moe_route(h: torch.Tensor, g: torch.Tensor, wg: torch.Tensor, M: int,
              topk: int, idx: torch.Tensor, w: torch.Tensor,
              dense: torch.Tensor | None = None, eps: float = 1e-5):
    """Fused MoE router (Mixtral semantics): per row RMSNorm(h)*g ->
    E dots vs wg[E,H] (f32) -> softmax -> top-k renormalized.
    idx: (M*topk,) int32; w: (M*topk,) f32; dense: (M*E,) f32 per-expert
    weights (0 if unrouted)."""
    E, H = wg.shape
    assert idx.numel() >= M * topk and w.numel() >= M * topk
    if dense is not None:
        assert dense.numel() >= M * E
    _check(lib().launch_moe_route(
        _ptr(h), _ptr(g), _ptr(wg), M, H, E, topk, ctypes.c_float(eps),
        _ptr(idx), _ptr(w), _ptr(dense), _stream()), "moe_route")


def expert_sort(idx: torch.Tensor, out: torch.Tensor, pairs: int, E: int):
    """Pairs (token, choice) by expert and the row tiles of each, for
    expert_gemm; out: int32, pairs * 1.2 + 4 E + 64 will do."""
    _check(lib().launch_expert_sort(
        _ptr(idx), _ptr(out), pairs, E, ctypes.c_long(out.numel()),
        _stream()), "expert_sort")


def expert_gemm(x: torch.Tensor, w: torch.Tensor, y: torch.Tensor,
                order: torch.Tensor, pairs: int, E: int, top: int, K: int,
                gather: bool, act: int = -1, sx: torch.Tensor | None = None,
                sw: torch.Tensor | None = None):
    """Each pair's row times its expert's W (w: experts one after the
    other; act: gate and up rows).  gather: x by token, y in ``order``; else
    x in ``order``, y by pair.  sx/sw: e4m3 rows and weights."""
    N = w.shape[0] // E // (2 if act >= 0 else 1)
    _check(lib().launch_expert_gemm(
        _ptr(x), _ptr(w), _ptr(sx), _ptr(sw), _ptr(y), _ptr(order), pairs, E,
        top, int(gather), N, K, act, _stream()), "expert_gemm")


def expert_gemm_plan(kind: str, pairs: int, E: int, N: int, K: int,
                     act: int = -1) -> dict:
    """Rows of expert_gemm's tiles and whether two groups of waves take turns at
    them (wide).  Host arithmetic only."""
    out = (ctypes.c_int * 2)()
    _check(lib().expert_gemm_plan(
        ("bf16", "fp8").index(kind), pairs, E, N, K, act,
        ctypes.cast(out, ctypes.c_void_p)), "expert_gemm_plan")
    return dict(rows=out[0], wide=bool(out[1]))


def expert_sum(y: torch.Tensor, w: torch.Tensor, idx: torch.Tensor,
               h: torch.Tensor, M: int, top: int):
    """h[t] += w[t, j] * y[t, j] over a token's choices, by expert."""
    _check(lib().launch_expert_sum(
        _ptr(y), _ptr(w), _ptr(idx), _ptr(h), M, top, h.shape[-1], _stream()),
        "expert_sum")


def moe_scale_add(y: torch.Tensor, x: torch.Tensor, w: torch.Tensor,
                  wstride: int, M: int, H: int):
    """y[m, :H] += w[m * wstride] * x[m, :H] (bf16, f32 math)."""
    _check(lib().launch_moe_scale_add(
        _ptr(y), _ptr(x), _ptr(w), ctypes.c_long(wstride), M, H,
        _stream()), "moe_scale_add")
