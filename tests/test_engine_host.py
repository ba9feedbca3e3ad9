"""The engine's choices on the host, without a GPU: what goes to which
kernel with which arguments."""

import os
import re
import types

import numpy as np
import pytest
import torch

from llm_np_cp_amd.models import decode_loop
from llm_np_cp_amd.models import engine as eng


class Calls(list):
    def __getattr__(self, name):
        def call(*a, **k):
            self.append((name, a, k))
        return call


def fake(**kw):
    """What _rows and _linear read of an engine."""
    m = types.SimpleNamespace(
        config=types.SimpleNamespace(rms_norm_eps=1e-5), fp8=False,
        wq4=False, b_gemm_acc=None, row_cnt=None, tile_cnt=None,
        b_xn=torch.zeros(32, 64), b_xq=torch.zeros(32 * 64),
        b_sx=torch.zeros(32))
    m.__dict__.update(kw)
    m._rows = types.MethodType(eng.GPUModel._rows, m)
    return m


@pytest.mark.parametrize("M", [1, 3, 16, 17])
@pytest.mark.parametrize("fp8", [False, True])
def test_linear_passes_bias_and_gate_on(monkeypatch, M, fp8):
    calls = Calls()
    calls.FEW_ROWS, calls.ROW_NORM_K = 16, 4096
    monkeypatch.setattr(eng, "ho", calls)
    x, y, b = torch.zeros(32, 64), torch.zeros(32, 64), torch.zeros(64)
    w = torch.zeros(128, 64)
    lw = {"w": w, "w_q": w, "w_s": torch.zeros(128)}
    eng.GPUModel._linear(fake(fp8=fp8), lw, "w", x, y, M=M, bias=b, act=1)
    name, _, kw = calls[-1]
    assert name == ("gemm_fp8" if fp8 else "gemm") if M > 16 else \
        ("gemv_fp8" if fp8 and M == 1 else "row_gemm")
    assert (kw["res"] if name == "gemv_fp8" else kw["bias"]) is b
    assert kw["act"] == 1 and kw.get("glu", True)


def test_linear_refuses_what_a_path_cannot_add(monkeypatch):
    calls = Calls()
    calls.FEW_ROWS, calls.ROW_NORM_K = 16, 4096
    monkeypatch.setattr(eng, "ho", calls)
    x, w = torch.zeros(32, 64), torch.zeros(128, 64)
    lw = {"w_q": w, "w_s": w, "w_q4": w, "w_e4": w}
    with pytest.raises(AssertionError):         # one row: one of them
        eng.GPUModel._linear(fake(fp8=True), lw, "w", x, x, M=1, res=x,
                             bias=x[0])
    with pytest.raises(AssertionError):         # gate and up apart
        eng.GPUModel._linear(fake(fp8=True, wq4=True), lw, "w", x, x, M=20,
                             res=x, act=0)
    assert not calls


def test_every_header_is_known_to_the_build():
    from csrc.build import CSRC, HEADERS, LIBS

    there = [f for f in os.listdir(CSRC) if f.endswith((".h", ".hip"))]
    names = {n for f in there for n in re.findall(
        r'#include "(.+?)"', open(os.path.join(CSRC, f)).read())}
    assert names <= set(HEADERS) <= set(there)
    assert {s for src in LIBS.values() for s in src} <= set(there)


def test_asm_that_sets_m0_says_so():
    """LDS loads of builtins go by m0 too, and the compiler keeps it."""
    from csrc.build import CSRC

    found = 0
    for f in os.listdir(CSRC):
        if f.endswith((".h", ".hip")):
            text = open(os.path.join(CSRC, f)).read()
            for asm in re.findall(r"\basm\b[^(]*\((.*?)\);", text, re.S):
                if re.search(r"\bs_mov_b32 m0\b", asm):
                    found += 1
                    assert '"m0"' in asm, f
    assert found


# one piece of any shape: rows follow one another; parts of a fused row: they
# are as far apart as it is long (a single row may say anything)
def test_distance_of_rows():
    from llm_np_cp_amd.ops.hip_ops import _ld

    M, nh, kvh, hd = 5, 4, 2, 16
    q = torch.zeros(M, nh * hd)
    for shape in ((M, nh * hd), (M * nh * hd,), (M, nh, hd), (1, M, nh, hd),
                  (1, M * nh * hd), (M * nh, hd)):
        assert _ld(q.view(shape), nh * hd) == nh * hd
    fused = torch.zeros(M, (nh + 2 * kvh) * hd)
    for t, w in zip(fused.split([nh * hd, kvh * hd, kvh * hd], 1),
                    (nh * hd, kvh * hd, kvh * hd)):
        assert _ld(t, w) == fused.shape[1]


# the first of a longer list of experts, unless there are rows for more
@pytest.mark.parametrize("listed,rows,glu,taken", [
    (1, 1, False, 1), (3, 1, False, 1), (3, 3, False, 3), (9, 2, False, 2),
    (3, 1, True, 1), (2, 2, True, 2), (2, 5, True, 2)])
def test_experts_there_are_rows_for(monkeypatch, listed, rows, glu, taken):
    from llm_np_cp_amd.ops import hip_ops as ho

    N, K, args = 32, 64, []
    lib = types.SimpleNamespace(
        launch_gemv=lambda *a: args.append(dict(zip(range(99), a))) or 0)
    monkeypatch.setattr(ho, "lib", lambda: lib)
    monkeypatch.setattr(ho, "_stream", lambda: 0)
    x, y = torch.zeros(1 if glu else rows, K), torch.zeros(rows if glu else 1, N)
    W = torch.zeros(N * (2 if glu else 1), K)
    idx, p = torch.zeros(listed, dtype=torch.int32), torch.zeros(listed)
    ho.gemv(W, x, y, eidx=idx, wstride=N * K, oscale=p, glu=glu)
    assert args[0][22] == taken and args[0][10] == N and args[0][11] == K


class Loop(decode_loop.DecodeLoop):
    max_seq = 1000

    def __init__(self):
        self.sizes = []

    def prefill(self, ids):
        pass

    def decode(self, n, **kw):
        self.sizes.append(n)
        return np.arange(n)


@pytest.mark.parametrize("kw,sizes", [
    (dict(), [256, 44]), (dict(chunk=8), [8] * 37 + [4]),
    (dict(chunk=100), [100, 100, 100]), (dict(chunk=300), [300]),
    (dict(on_ids=lambda ids: None), [16] * 18 + [12]),
    (dict(eos_id=999), [16] * 18 + [12]),
    (dict(eos_id=[999], chunk=150), [150, 150]),
    (dict(stop_fn=lambda ids: len(ids) >= 40), [16] * 3)])
def test_tokens_are_fetched_in_the_chunks_asked_for(kw, sizes):
    m = Loop()
    assert len(m.generate_tokens([1, 2], 300, **kw)) == sum(sizes)
    assert m.sizes == sizes


# a block of 256 dims has a CU to itself, one for every four query heads of a kv
# head; of other dims two share one and heads are not counted
@pytest.mark.parametrize("hd,nh,kvh,rows,most,ranges", [
    (256, 8, 1, 16, 16, 8), (256, 8, 1, 32, 8, 4), (256, 8, 1, 64, 64, 2),
    (256, 8, 1, 200, 64, 1), (256, 4, 1, 16, 64, 16), (256, 16, 8, 16, 64, 2),
    (256, 20, 4, 8, 64, 4), (256, 8, 4, 1, 20, 20), (128, 8, 1, 16, 64, 16),
    (64, 32, 4, 16, 64, 4)])
def test_ranges_of_a_step(hd, nh, kvh, rows, most, ranges):
    m = types.SimpleNamespace(hd=hd, nh_l=nh, kvh_l=kvh, attn_split=most)
    assert eng.GPUModel._ranges(m, rows) == ranges
