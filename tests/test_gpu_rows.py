"""Kernels for rows of a prompt or a group: the edges of their tiles."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def normal(*shape, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(*shape, generator=g, device="cuda") *
            scale).bfloat16()


def off(y, ref):
    """2-norm of the difference over that of the reference."""
    return ((y.double() - ref).norm() / ref.norm()).item()


def e4m3(x):
    """Rows of the last axis scaled to 448: bytes, scales, their values."""
    s = x.float().abs().amax(-1).clamp(min=1e-8) / 448
    q = (x.float() / s[..., None]).to(torch.float8_e4m3fn)
    return (q.view(torch.uint8).contiguous(), s.contiguous(),
            q.double() * s[..., None].double())


# rows of a kv head: one short of, at and past 32 (one wave) and 128 (four);
# keys: a partial tile, a window inside one, enough to be split
@pytest.mark.parametrize("hd,nh,kvh", [(64, 8, 2), (128, 3, 1), (256, 2, 2)])
@pytest.mark.parametrize("M,pos0,window,cap", [
    (1, 0, 0, 0.0), (2, 63, 0, 50.0), (5, 901, 0, 0.0), (8, 700, 40, 0.0),
    (11, 2000, 0, 0.0), (32, 0, 7, 0.0), (33, 1, 0, 0.0), (43, 3, 0, 50.0),
    (129, 64, 33, 0.0)])
@pytest.mark.parametrize("kv8", [False, True])
def test_prompt_attention(hd, nh, kvh, M, pos0, window, cap, kv8):
    from llm_np_cp_amd.ops import hip_ops as ho

    T = pos0 + M
    q = normal(M, nh, hd, seed=1, scale=2.0)
    K, V = (normal(kvh, T + 3, hd, seed=s) for s in (2, 3))
    kS = vS = None
    Kd, Vd = K.double(), V.double()
    if kv8:
        (K, kS, Kd), (V, vS, Vd) = e4m3(K), e4m3(V)
    out = torch.full((M + 1, nh * hd), 7.0, device="cuda").bfloat16()
    part = torch.zeros(1 << 22, device="cuda")
    ho.attn_prefill_mfma(
        q, K, V, out, torch.tensor([pos0], dtype=torch.int32, device="cuda"),
        M, nh, kvh, hd, hd ** -0.5, softcap=cap, window=window, kS=kS, vS=vS,
        part=part, keys=T)
    i = pos0 + torch.arange(M, device="cuda")[:, None]
    j = torch.arange(T, device="cuda")
    bad = (j > i) | ((j <= i - window) if window else False)
    ref = torch.empty(M, nh, hd, dtype=torch.float64, device="cuda")
    for h in range(nh):
        s = q[:, h].double() @ Kd[h * kvh // nh, :T].T * hd ** -0.5
        s = cap * torch.tanh(s / cap) if cap else s
        p = torch.softmax(s.masked_fill(bad, -math.inf), -1)
        ref[:, h] = p @ Vd[h * kvh // nh, :T]
    # bf16 probabilities and results: 2^-9 at most each
    assert off(out[:M], ref.view(M, -1)) < 2.0 ** -8
    assert (out[M] == 7.0).all()
