#!/usr/bin/env python3
"""Per-kernel microbenchmark (runs on an MI355X box).

Times each decode-path kernel shape standalone: a hipGraph of REPS
launches, timed with CUDA events, reported as us/launch and effective
TB/s of weight traffic (small shapes stay in the caches; --layersim
times whole layers from memory).
"""

import os
import sys
import time

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

import torch  # noqa: E402


def time_graph(fn, reps=50, warmup=20):
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(3):
            fn()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(reps):
            fn()
    for _ in range(warmup):
        pass
    g.replay()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(5):
        g.replay()
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / (5 * reps)
    return dt * 1e6  # us per launch


def main():
    from csrc.build import ensure_built
    ensure_built()
    from llm_np_cp_amd.ops import hip_ops as ho

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)

    shapes = [
        ("qkv", 3072, 2048), ("wo", 2048, 2048), ("wgu", 16384, 2048),
        ("wdown", 2048, 8192), ("lm_head", 128256, 2048),
        ("9b_qkv", 8192, 3584), ("9b_wgu", 28672, 3584),
        ("huge", 262144, 2048),  # 1 GB bf16 > L3: honest HBM number
    ]
    print(f"{'shape':>9} {'N':>7} {'K':>6} | " +
          " | ".join(f"{v:>12}" for v in
                     ["bf16", "bf16 norm", "fp8", "fp8 norm"]))
    for name, N, K in shapes:
        W = torch.randn(N, K, device=dev).to(torch.bfloat16) * 0.05
        s = W.float().abs().amax(dim=1).clamp_min(1e-8) / 448.0
        Wq = (W.float() / s[:, None]).to(torch.float8_e4m3fn).view(torch.uint8)
        x = torch.randn(K, device=dev).to(torch.bfloat16)
        y = torch.empty(N, dtype=torch.bfloat16, device=dev)
        res = []
        g = torch.rand(K, device=dev)
        norm = dict(stage=ho.STAGE_NORM, g=g)
        for kind, kw in (("bf16", {}), ("bf16", norm), ("fp8", {}),
                         ("fp8", norm)):
            if kind == "bf16":
                fn = lambda: ho.gemv(W, x, y, **kw)
                nbytes = N * K * 2
            else:
                fn = lambda: ho.gemv_fp8(Wq, s, x, y, **kw)
                nbytes = N * K
            us = time_graph(fn)
            res.append(f"{us:6.2f}us {nbytes/us/1e6:5.2f}T")
        print(f"{name:>9} {N:>7} {K:>6} | " + " | ".join(f"{r:>12}" for r in res))

    # attention decode at several context lengths
    print("\nattn_dec (nh=32 kvh=8 hd=64):")
    nh, kvh, hd, S = 32, 8, 64, 8192
    kc = torch.randn(kvh, S, hd, device=dev).to(torch.bfloat16)
    vc = torch.randn_like(kc)
    qkv = torch.randn((nh + 2 * kvh) * hd, device=dev).to(torch.bfloat16)
    out = torch.empty(nh * hd, dtype=torch.bfloat16, device=dev)
    inv = 1.0 / (10000.0 ** (torch.arange(0, hd, 2).float() / hd))
    fr = torch.outer(torch.arange(S).float(), inv)
    cos_t = torch.cos(fr).to(dev)
    sin_t = torch.sin(fr).to(dev)
    for split in [1, 4, 8, 16]:
        scratch = torch.zeros(nh * split * (hd + 2), dtype=torch.float32,
                              device=dev)
        cnt = torch.zeros(nh, dtype=torch.int32, device=dev)
        for T in [128, 512, 2048, 8000]:
            pos = torch.tensor([T - 1], dtype=torch.int32, device=dev)
            us = time_graph(lambda: ho.attn_dec(
                qkv, kc, vc, out, pos, cos_t, sin_t, scratch, cnt,
                nh, kvh, hd, hd ** -0.5, split=split))
            print(f"  split={split:2d} T={T:5d}: {us:6.2f}us")

    # rmsnorm / sampler
    H = 2048
    xh = torch.randn(H, device=dev).to(torch.bfloat16)
    gh = torch.randn(H, device=dev)
    yh = torch.empty_like(xh)
    print(f"\nrmsnorm H={H}: {time_graph(lambda: ho.rmsnorm(xh, gh, yh)):.2f}us")

    V = 128256
    logits = torch.randn(V, device=dev)
    ctr = torch.zeros(1, dtype=torch.int64, device=dev)
    gmax = torch.zeros(1, dtype=torch.int64, device=dev)
    pick = torch.zeros(1, dtype=torch.int64, device=dev)
    nt_ = torch.zeros(1, dtype=torch.int32, device=dev)
    ring = torch.zeros(65536, dtype=torch.int32, device=dev)
    nout = torch.zeros(1, dtype=torch.int32, device=dev)
    ln = torch.zeros(1, dtype=torch.int32, device=dev)
    us = time_graph(lambda: ho.sample(logits, 0.1, True, 0, ctr, gmax, pick,
                                      nt_, ring, nout, ln))
    print(f"sample greedy V={V}: {us:.2f}us")
    us = time_graph(lambda: ho.sample(logits, 0.1, False, 0, ctr, gmax, pick,
                                      nt_, ring, nout, ln))
    print(f"sample min-p  V={V}: {us:.2f}us")


if __name__ == "__main__" and "--layersim" not in sys.argv:
    main()


def layersim():
    """In-context layer simulation: a graph over 16 DISTINCT layers'
    GEMV weights (2.4 GB total > L3), the products of a decode step as the
    engine launches them — honest per-layer time without the full engine;
    with all blocks and with half of them."""
    from csrc.build import ensure_built
    ensure_built()
    from llm_np_cp_amd.ops import hip_ops as ho

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    H, I, NKV = 2048, 8192, 1024
    L = 16
    layers = []
    for _ in range(L):
        layers.append(dict(
            wqkv=torch.randn(H + NKV, H, device=dev).to(torch.bfloat16),
            wo=torch.randn(H, H, device=dev).to(torch.bfloat16),
            wgu=torch.randn(2 * I, H, device=dev).to(torch.bfloat16),
            wdown=torch.randn(H, I, device=dev).to(torch.bfloat16),
        ))
    h = torch.randn(H, device=dev).to(torch.bfloat16)
    qkv = torch.empty(H + NKV, dtype=torch.bfloat16, device=dev)
    att = torch.randn(H, device=dev).to(torch.bfloat16)
    act = torch.empty(I, dtype=torch.bfloat16, device=dev)
    g1 = torch.randn(H, device=dev)

    def one_pass(cap, **norm):
        for lw in layers:
            ho.gemv(lw["wqkv"], h, qkv, maxblocks=cap, **norm)
            ho.gemv(lw["wo"], att, h, res=h, maxblocks=cap)
            ho.gemv(lw["wgu"], h, act, glu=True, maxblocks=cap, **norm)
            ho.gemv(lw["wdown"], act, h, res=h, maxblocks=cap)

    print("layersim: 16 llama-1b layers of GEMVs (121.6 MB/layer bf16)")
    # without the norms: what their staging costs beside the stream
    for name, norm in (("staged", dict(stage=ho.STAGE_NORM, g=g1)),
                       ("all-raw", {})):
        for cap in (0, 128):
            us = time_graph(lambda: one_pass(cap, **norm), reps=5, warmup=5)
            print(f"  {name} cap={cap:5d}: {us/L:7.2f}us/layer "
                  f"({121.6e6*L/us/1e6:4.2f} TB/s)")


if __name__ == "__main__" and "--layersim" in sys.argv:
    layersim()
    sys.exit(0)
