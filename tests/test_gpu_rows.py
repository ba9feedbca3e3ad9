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
# keys: a partial tile, a window inside one, enough to be split, into parts of
# one tile and of some
@pytest.mark.parametrize("hd,nh,kvh", [(64, 8, 2), (128, 3, 1), (256, 2, 2)])
@pytest.mark.parametrize("M,pos0,window,cap", [
    (1, 0, 0, 0.0), (2, 63, 0, 50.0), (5, 901, 0, 0.0), (8, 700, 40, 0.0),
    (11, 2000, 0, 0.0), (32, 0, 7, 0.0), (33, 1, 0, 0.0), (43, 3, 0, 50.0),
    (129, 64, 33, 0.0), (64, 2000, 0, 0.0), (90, 500, 300, 50.0),
    (300, 100, 0, 0.0)])
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


# blocks of which two groups of waves take the keys in turn: up to a block a CU
# and more, first rows with one tile of keys (the second group has none), an odd
# number, keys ahead of the rows, windows, a cap; rows that end inside a wave.
# And as many blocks whose way is another: one tile in all, ranges, 256 dims,
# e4m3 keys of 64
@pytest.mark.parametrize("hd,nh,kvh,M,pos0,window,cap,kv8", [
    (64, 80, 80, 50, 0, 0, 0.0, False), (64, 32, 8, 333, 0, 0, 0.0, False),
    (64, 32, 8, 611, 70, 0, 30.0, False), (64, 40, 8, 1037, 0, 0, 0.0, False),
    (64, 32, 8, 500, 300, 200, 0.0, False),
    (64, 32, 8, 611, 0, 0, 0.0, True),
    (128, 72, 72, 64, 0, 0, 0.0, False), (128, 32, 8, 430, 0, 0, 0.0, False),
    (128, 16, 4, 1100, 33, 0, 50.0, False), (128, 24, 8, 1450, 0, 0, 0.0, False),
    (128, 32, 8, 480, 100, 130, 0.0, False),
    (128, 32, 8, 430, 5, 0, 0.0, True), (128, 24, 8, 1450, 0, 0, 0.0, True),
    (256, 16, 8, 601, 0, 0, 50.0, False)])
def test_prompt_attention_of_many_blocks(hd, nh, kvh, M, pos0, window, cap,
                                         kv8):
    test_prompt_attention(hd, nh, kvh, M, pos0, window, cap, kv8)


# the same of several sequences, of ragged lengths, one of them behind keys of its
# own: up to a block a CU and more, sequences that leave the second group without
# a tile, windows, a cap, pools out of order
@pytest.mark.parametrize("hd,nh,kvh,segs,window,cap,kv8", [
    (64, 32, 8, [(2, 0, 333), (0, 70, 301), (1, 0, 65)], 0, 0.0, False),
    (64, 32, 8, [(2, 0, 533), (0, 70, 301), (1, 0, 5)], 470, 30.0, False),
    (64, 40, 8, [(2, 0, 640), (0, 0, 410), (1, 100, 33)], 520, 0.0, False),
    (64, 72, 8, [(0, 0, 300), (2, 300, 250), (1, 0, 2)], 0, 50.0, False),
    (128, 16, 4, [(0, 0, 600), (1, 30, 60), (2, 0, 3)], 0, 0.0, False),
    (128, 12, 2, [(1, 0, 900), (0, 300, 60), (2, 0, 40)], 0, 50.0, False),
    (128, 64, 8, [(1, 0, 650), (0, 600, 101), (2, 0, 17)], 0, 0.0, False),
    (128, 64, 8, [(1, 0, 750), (0, 0, 101), (2, 0, 17)], 700, 0.0, False),
    (128, 32, 8, [(2, 0, 333), (0, 70, 301), (1, 0, 65)], 200, 0.0, True),
    (128, 64, 8, [(1, 0, 450), (0, 600, 101), (2, 0, 17)], 0, 30.0, True)])
def test_prompts_of_one_batch_by_two_groups_of_waves(hd, nh, kvh, segs, window,
                                                     cap, kv8):
    from llm_np_cp_amd.ops import hip_ops as ho

    M, keys = sum(n for _, _, n in segs), max(p + n for _, p, n in segs)
    most, S = max(n for _, _, n in segs), keys + 3
    tiles = torch.from_numpy(ho.attn_tiles(segs, nh // kvh)).cuda()
    assert ho.attn_prefill_plan(M, nh, kvh, hd, keys, window, kv8, 1 << 22,
                                most, len(tiles))["two"]
    q = normal(M, nh, hd, seed=1, scale=2.0)
    K, V = (normal(3, kvh, S, hd, seed=s) for s in (2, 3))
    kS = vS = None
    Kd, Vd = K.double(), V.double()
    if kv8:
        (K, kS, Kd), (V, vS, Vd) = e4m3(K), e4m3(V)
    out = torch.full((M + 1, nh * hd), 7.0, device="cuda").bfloat16()
    ho.attn_prefill_mfma(
        q, K, V, out, None, M, nh, kvh, hd, hd ** -0.5, softcap=cap,
        window=window, kS=kS, vS=vS, part=torch.zeros(1 << 22, device="cuda"),
        keys=keys, tiles=tiles, most=most)
    ref, at = torch.empty(M, nh, hd, dtype=torch.float64, device="cuda"), 0
    for b, p, n in segs:
        i = p + torch.arange(n, device="cuda")[:, None]
        j = torch.arange(p + n, device="cuda")
        bad = (j > i) | ((j <= i - window) if window else False)
        for h in range(nh):
            g = h * kvh // nh
            s = q[at:at + n, h].double() @ Kd[b, g, :p + n].T * hd ** -0.5
            s = cap * torch.tanh(s / cap) if cap else s
            w = torch.softmax(s.masked_fill(bad, -math.inf), -1)
            ref[at:at + n, h] = w @ Vd[b, g, :p + n]
        # bf16 probabilities and results: 2^-9 at most each
        assert off(out[at:at + n], ref[at:at + n].view(n, -1)) < 2.0 ** -8
        at += n
    assert (out[M] == 7.0).all()


# parts of the keys in lines, 16 rows a block of their sum: rows that end inside
# one and with one, fewer parts than are on the way together (eight), as many, one
# more; and row by row, also as few rows as that goes by
@pytest.mark.parametrize("hd,nh,kvh,M,pos0,window,cap,ranges,by_row", [
    (64, 4, 2, 67, 220, 0, 0.0, 5, False), (64, 8, 2, 300, 2000, 0, 0.0, 9, False),
    (64, 4, 4, 400, 900, 0, 30.0, 7, False), (128, 3, 1, 43, 190, 0, 0.0, 4, False),
    (128, 8, 1, 144, 300, 0, 0.0, 7, False), (128, 6, 2, 400, 900, 700, 0.0, 6, False),
    (256, 2, 2, 130, 30, 0, 50.0, 5, False), (256, 4, 1, 330, 200, 0, 0.0, 9, False),
    (256, 8, 1, 200, 500, 0, 0.0, 8, False), (64, 9, 3, 21, 1800, 0, 0.0, 28, True),
    (128, 4, 2, 210, 800, 0, 0.0, 8, True), (256, 4, 1, 270, 700, 0, 0.0, 11, True)])
@pytest.mark.parametrize("kv8", [False, True])
def test_prompt_attention_in_parts(hd, nh, kvh, M, pos0, window, cap, ranges,
                                   by_row, kv8):
    from llm_np_cp_amd.ops import hip_ops as ho

    p = ho.attn_prefill_plan(M, nh, kvh, hd, pos0 + M, window, kv8, 1 << 22)
    if not kv8:
        assert p == dict(ranges=ranges, two=False, by_row=by_row)
    test_prompt_attention(hd, nh, kvh, M, pos0, window, cap, kv8)


# a part of the keys whose weight beside the others' underflows, with values
# that are no number: as in one softmax, 0 times them is none either
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_prompt_attention_without_a_number(hd):
    from llm_np_cp_amd.ops import hip_ops as ho

    M, pos0, nh, kvh = 5, 901, 4, 2
    T = pos0 + M
    q = torch.ones(M, nh, hd, device="cuda").bfloat16()
    K, V = (normal(kvh, T, hd, seed=s) for s in (2, 3))
    K[:, :128] = -40.0
    V[:, 10, 3], V[:, 70, 5] = math.nan, math.inf
    out = torch.empty(M, nh, hd, device="cuda").bfloat16()
    ho.attn_prefill_mfma(
        q, K, V, out, torch.tensor([pos0], dtype=torch.int32, device="cuda"),
        M, nh, kvh, hd, hd ** -0.5,
        part=torch.zeros(1 << 22, device="cuda"), keys=T)
    bad = out.isnan()
    assert bad[..., 3].all() and bad[..., 5].all()
    bad[..., 3] = bad[..., 5] = False
    assert not bad.any()


def mxfp4_values(q, e):
    """MXFP4 bytes and exponents as 64-bit values."""
    grid = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0],
                        dtype=torch.float64, device=q.device)
    c = torch.stack([q & 15, q >> 4], -1).reshape(q.shape[0], -1).long()
    v = grid[c & 7] * torch.where(c > 7, -1.0, 1.0)
    return v * torch.exp2(e.double() - 127).repeat_interleave(32, 1)


# outputs: less than half a tile, a tile and a rest, more tiles than blocks;
# K: one slab of 64, slabs that eight waves share unevenly, split over blocks;
# more outputs than LDS has room for the sums of beside 16 long rows
@pytest.mark.parametrize("N,K", [(5, 64), (24, 192), (200, 320), (520, 8192),
                                 (4616, 1088), (30000, 4608)])
@pytest.mark.parametrize("M", [1, 7, 16])
@pytest.mark.parametrize("kind", ["bf16", "fp8", "fp4"])
@pytest.mark.parametrize("norm,act", [(False, -1), (True, -1), (False, 1),
                                      (True, 0)])
def test_few_rows(N, K, M, kind, norm, act):
    from llm_np_cp_amd.ops import hip_ops as ho

    if norm and K > ho.ROW_NORM_K:
        pytest.skip("normed by a kernel of its own")
    W = normal(N * (2 if act >= 0 else 1), K, seed=4, scale=K ** -0.5)
    X = normal(M, K + 16, seed=5)[:, :K]            # rows apart
    g = torch.rand(K, device="cuda") + 0.5 if norm else None
    bias, res = (normal(M, N, seed=6) for _ in range(2))
    kw, Wd, x = {}, W.double(), X.double()
    if norm:
        x = x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-5) * g.double()
    if kind == "fp8":
        W, kw["ws"], Wd = e4m3(W)
        q, s, x = e4m3(x)
        if not norm:
            X, kw["sx"] = q, s
    elif kind == "fp4":
        q = torch.empty(W.shape[0], K // 2, dtype=torch.uint8, device="cuda")
        e = torch.empty(W.shape[0], K // 32, dtype=torch.uint8, device="cuda")
        ho.quant_fp4(W, q, e)
        W, kw["we"], Wd = q, e, mxfp4_values(q, e)
    part = torch.zeros(1 << 22, device="cuda")
    cnt = torch.zeros(256, dtype=torch.int32, device="cuda")
    Y = torch.full((M + 1, N), 7.0, device="cuda").bfloat16()
    for _ in range(2):                              # counters are left zero
        ho.row_gemm(X, W, Y, M, g=g, bias=bias[0].contiguous(), res=res,
                    act=act, softcap=30.0, part=part, cnt=cnt, **kw)
    z = x @ Wd.T
    if kind == "fp8" and act >= 0:
        z = z.bfloat16().double()
    if act >= 0:
        f = (torch.nn.functional.silu if act == 0 else lambda t:
             torch.nn.functional.gelu(t, approximate="tanh"))
        z = f(z[:, :N]) * z[:, N:]
    z = 30.0 * torch.tanh(z / 30.0) + bias[0].double() + res.double()
    # bf16 normed rows and results: 2^-9 at most each, twice through a gate;
    # a normed value that lies on the edge of two e4m3 ones may take the
    # other: 2^-4 of it, and one in some hundred does
    assert off(Y[:M], z) < (2.0 ** -6 if norm and kind == "fp8"
                            else 2.0 ** -7)
    assert (Y[M] == 7.0).all() and not cnt.any()


# the rows that an e4m3 product makes for itself: a prompt's by way of bf16, a
# step's from fp32.  A unit matrix shows them: exact in an fp32 result.
@pytest.mark.parametrize("K", [64, 512, 2304, 4096])
@pytest.mark.parametrize("M", [2, 16])
def test_rows_rounded_on_the_way(K, M):
    from llm_np_cp_amd.ops import hip_ops as ho

    W = torch.eye(K, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8)
    X, one = normal(M, K, seed=12), torch.ones(K, device="cuda")
    g = normal(1, K, seed=13)[0].float().abs() + 0.5
    x = X.double()
    x = (x * torch.rsqrt(x.pow(2).mean(1, keepdim=True) + 1e-5)
         * g.double()).abs()
    got = {}
    for norm16 in (False, True):
        Y = torch.full((M + 1, K), 7.0, device="cuda")
        ho.row_gemm(X, W, Y, M, ws=one, g=g, norm16=norm16)
        # The norm's sums and products in fp32, the scale and the division by
        # it are off by less than 2^-18 (33 roundings of a sum of squares,
        # halved by the root, and a dozen more): a value on an edge of bf16
        # or e4m3 may take either side, no other may.
        lo, hi = (x * (1 - 2.0 ** -18)).float(), (x * (1 + 2.0 ** -18)).float()
        if norm16:
            lo, hi = lo.bfloat16().float(), hi.bfloat16().float()
        slo, shi = (v.amax(1, keepdim=True) / 448 for v in (lo, hi))
        most = torch.full_like(hi, 448.0)       # of e4m3
        lo = (lo / shi * (1 - 2.0 ** -18)).to(torch.float8_e4m3fn).float()
        hi = torch.minimum(hi / slo * (1 + 2.0 ** -18), most)
        hi = hi.to(torch.float8_e4m3fn).float()
        y = Y[:M].abs()
        assert (y >= lo * slo * (1 - 2.0 ** -18)).all()
        assert (y <= hi * shi * (1 + 2.0 ** -18)).all()
        assert ((Y[:M] >= 0) == (X >= 0))[y > 0].all()
        assert (Y[M] == 7.0).all()
        got[norm16] = Y[:M]
    if M * K > 8192:                    # and the two are told apart
        d = (got[True] - got[False]).abs() > got[False].abs() * 2.0 ** -6
        assert d.float().mean() > 0.008


# what a step's gate hands to the rounding behind it: fp32, from bf16 halves
@pytest.mark.parametrize("N,K", [(24, 192), (520, 8192)])
@pytest.mark.parametrize("M", [3, 16])
def test_gate_in_fp32(N, K, M):
    from llm_np_cp_amd.ops import hip_ops as ho

    (W, ws, Wd) = e4m3(normal(2 * N, K, seed=4, scale=K ** -0.5))
    X, sx, x = e4m3(normal(M, K, seed=5))
    part = torch.zeros(1 << 20, device="cuda")
    cnt = torch.zeros(256, dtype=torch.int32, device="cuda")
    Y = torch.full((M + 1, N), 7.0, device="cuda")
    for _ in range(2):
        ho.row_gemm(X, W, Y, M, ws=ws, sx=sx, act=1, part=part, cnt=cnt)
    z = (x @ Wd.T).bfloat16().double()
    z = torch.nn.functional.gelu(z[:, :N], approximate="tanh") * z[:, N:]
    # A half takes the other of two bf16 values where its sum, at most
    # K 2^-24 off, crosses the middle of their distance of 2^-8: one in eight
    # for 8192, some hundred times fewer by chance.  All others are fp32's; a
    # result in bf16 would be off by 2^-9 nearly everywhere.
    far = (Y[:M] - z).abs() > z.abs() * 2.0 ** -14
    assert far.double().mean() < 1 / 16
    assert (Y[M] == 7.0).all() and not cnt.any()


# long rows beside room for parts of all, of fewer rows and of none; a tile of
# sums that just does not fit (8 rows of 9536)
@pytest.mark.parametrize("kind,M,N,K", [
    ("bf16", 16, 520, 8192), ("bf16", 8, 4608, 9536), ("fp8", 13, 300, 19008),
    ("fp4", 16, 70, 12288)])
@pytest.mark.parametrize("act", [-1, 0])
@pytest.mark.parametrize("room", [0, 100000, 1 << 22])
def test_few_rows_of_little_room(kind, M, N, K, act, room):
    from llm_np_cp_amd.ops import hip_ops as ho

    W = normal(N * (2 if act >= 0 else 1), K, seed=4, scale=K ** -0.5)
    X = normal(M, K + 16, seed=5)[:, :K]
    bias, res = (normal(M, N, seed=6) for _ in range(2))
    kw, Wd, x = {}, W.double(), X.double()
    if kind == "fp8":
        W, kw["ws"], Wd = e4m3(W)
        X, kw["sx"], x = e4m3(X)
    elif kind == "fp4":
        q = torch.empty(W.shape[0], K // 2, dtype=torch.uint8, device="cuda")
        e = torch.empty(W.shape[0], K // 32, dtype=torch.uint8, device="cuda")
        ho.quant_fp4(W, q, e)
        W, kw["we"], Wd = q, e, mxfp4_values(q, e)
    part = torch.full((room + 64,), 7.0, device="cuda")
    cnt = torch.zeros(256, dtype=torch.int32, device="cuda")
    Y = torch.full((M + 1, N), 7.0, device="cuda").bfloat16()
    Y[:M] = res                                     # in place
    ho.row_gemm(X, W, Y, M, bias=bias[0].contiguous(), res=Y, act=act,
                part=part[:room], cnt=cnt, **kw)
    z = x @ Wd.T
    if act >= 0:
        if kind == "fp8":
            z = z.bfloat16().double()
        z = torch.nn.functional.silu(z[:, :N]) * z[:, N:]
    z = z + bias[0].double() + res.double()
    # exact products, fp32 sums, bf16 results: 2^-9 at most, and the halves
    # of an e4m3 gate
    assert off(Y[:M], z) < 2.0 ** -8
    assert (Y[M] == 7.0).all() and not cnt.any() and (part[room:] == 7.0).all()


# tiles of 32 to 256 rows and 64 to 256 outputs, by what the sizes call for:
# a rest of a tile both ways, outputs that are no multiple of four, K of one
# slab, of one more than the buffers, split over blocks, half a slab (e4m3)
@pytest.mark.parametrize("M,N,K", [
    (17, 70, 64), (37, 258, 192), (33, 200, 8192), (130, 1000, 320),
    (300, 3000, 448), (310, 2500, 1216), (513, 4100, 256), (1030, 2050, 64),
    (2050, 6200, 128), (2049, 16500, 64)])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
@pytest.mark.parametrize("act", [-1, 0, 1])
def test_many_rows(M, N, K, kind, act):
    from llm_np_cp_amd.ops import hip_ops as ho

    W = normal(N * (2 if act >= 0 else 1), K, seed=7, scale=K ** -0.5)
    X = normal(M, K, seed=8)
    bias, res = normal(N, seed=9), normal(M, N, seed=10)
    part = torch.zeros(1 << 24, device="cuda")
    cnt = torch.zeros(1024, dtype=torch.int32, device="cuda")
    Y = torch.full((M + 1, N), 7.0, device="cuda").bfloat16()
    kw = dict(res=res, bias=bias, act=act, accbuf=part, cnt=cnt)
    Wd, x = W.double(), X.double()
    if kind == "fp8":
        (W, sw, Wd), (X, sx, x) = e4m3(W), e4m3(X)
    for _ in range(2):                              # counters are left zero
        if kind == "fp8":
            ho.gemm_fp8(X, sx, W, sw, Y[:M], M, K, **kw)
        else:
            ho.gemm(X, W, Y[:M], **kw)
    z = x @ Wd.T
    if act >= 0:
        if kind == "fp8":               # bf16 halves on their way to e4m3
            z = z.bfloat16().double()
        f = (torch.nn.functional.silu if act == 0 else lambda t:
             torch.nn.functional.gelu(t, approximate="tanh"))
        z = f(z[:, :N]) * z[:, N:]
    z = z + bias.double() + res.double()
    # exact products, fp32 sums, bf16 results: 2^-9 at most
    assert off(Y[:M], z) < 2.0 ** -9
    assert (Y[M] == 7.0).all() and not cnt.any()


# each tile (rows and outputs, parts of K, waves, whether by two groups of them) by
# itself and with K split over blocks, where the sizes above leave it out; 128x256
# of e4m3 rows with half a slab too, 128x128 of four waves and of eight
@pytest.mark.parametrize("M,N,K,kind,act,tile", [
    (1037, 10902, 192, "bf16", -1, (128, 128, 1, 4, False)),
    (525, 11405, 704, "bf16", -1, (128, 256, 1, 8, True)),
    (513, 3878, 512, "bf16", -1, (128, 64, 1, 8, False)),
    (1601, 598, 5632, "bf16", -1, (128, 128, 3, 8, False)),
    (132, 16809, 64, "bf16", -1, (64, 128, 1, 8, False)),
    (429, 376, 2112, "bf16", -1, (64, 64, 3, 8, False)),
    (66, 58, 896, "bf16", -1, (32, 64, 3, 4, False)),
    (517, 1812, 448, "bf16", 0, (128, 64, 1, 8, False)),
    (589, 418, 7552, "bf16", 0, (128, 128, 5, 8, False)),
    (130, 8243, 128, "bf16", 0, (64, 128, 1, 8, False)),
    (33, 8564, 6720, "bf16", 0, (64, 128, 3, 8, False)),
    (582, 1621, 1152, "bf16", 0, (64, 64, 1, 8, False)),
    (43, 65, 960, "bf16", 0, (32, 64, 1, 4, False)),
    (26, 129, 2112, "bf16", 0, (32, 64, 7, 4, False)),
    (584, 5294, 192, "fp8", -1, (128, 64, 1, 8, False)),
    (871, 4614, 448, "fp8", -1, (128, 64, 1, 8, False)),
    (425, 340, 6400, "fp8", -1, (64, 64, 5, 8, False)),
    (67, 70, 960, "fp8", -1, (32, 64, 1, 4, False)),
    (137, 7852, 448, "fp8", 0, (128, 64, 1, 8, False)),
    (596, 845, 7680, "fp8", 0, (128, 64, 3, 8, False)),
    (19, 16845, 64, "fp8", 0, (64, 128, 1, 8, False)),
    (378, 193, 5056, "fp8", 0, (32, 64, 2, 4, False)),
    (145, 16724, 448, "fp8", -1, (64, 128, 1, 8, False)),
    (174, 5488, 6464, "fp8", -1, (64, 128, 3, 8, False)),
    (98, 8286, 6464, "fp8", -1, (128, 64, 3, 8, False)),
    (68, 16752, 3264, "fp8", -1, (128, 128, 1, 8, False)),
    (99, 8213, 9600, "fp8", -1, (128, 128, 3, 8, False)),
    (200, 16680, 448, "fp8", -1, (128, 256, 1, 8, False)),
    (330, 3640, 19264, "fp8", -1, (128, 256, 5, 8, False)),
    (214, 2487, 9600, "fp8", 0, (128, 128, 3, 8, False)),
    (130, 6977, 4096, "fp8", 0, (128, 128, 1, 8, False)),
    (133, 12433, 448, "fp8", 0, (128, 256, 1, 8, False)),
    (335, 2003, 19264, "fp8", 0, (128, 256, 5, 8, False)),
    (166, 2812, 9600, "fp8", 0, (64, 128, 3, 8, False)),
    (66, 2853, 9600, "fp8", 0, (128, 64, 5, 8, False)),
    (67, 2744, 9600, "bf16", -1, (128, 64, 5, 8, False)),
    (66, 1512, 9600, "bf16", 0, (128, 64, 5, 8, False)),
    (69, 8808, 2112, "bf16", 0, (128, 128, 1, 8, False)),
    (35, 1835, 3264, "bf16", 0, (64, 64, 4, 8, False)),
    (905, 8494, 384, "bf16", -1, (64, 64, 1, 8, False)),
    (391, 10822, 192, "bf16", -1, (128, 128, 1, 4, False)),
    (1045, 11186, 192, "bf16", -1, (128, 128, 1, 4, False)),
    (675, 10949, 320, "bf16", -1, (64, 64, 1, 8, False)),
    (199, 8994, 8192, "bf16", -1, (128, 128, 1, 8, False)),
    (385, 8380, 64, "bf16", 0, (64, 128, 1, 8, False)),
    (1188, 9848, 64, "bf16", 0, (128, 128, 1, 4, False)),
    (1159, 9732, 128, "bf16", 0, (128, 128, 1, 4, False)),
    (1052, 10895, 192, "bf16", 0, (128, 64, 1, 8, False)),
    (259, 8593, 128, "bf16", 0, (64, 128, 1, 8, False)),
    (566, 10887, 128, "bf16", 0, (128, 128, 1, 4, False)),
    (555, 11005, 192, "bf16", 0, (128, 64, 1, 8, False)),
    (1167, 9842, 128, "fp8", 0, (64, 128, 1, 8, False)),
    (1164, 9823, 256, "fp8", 0, (128, 64, 1, 8, False)),
    (1156, 10068, 384, "fp8", 0, (64, 128, 1, 8, False)),
    (547, 11509, 128, "fp8", 0, (64, 128, 1, 8, False)),
    (542, 11246, 256, "fp8", 0, (128, 64, 1, 8, False)),
    (521, 11510, 384, "fp8", 0, (128, 64, 1, 8, False))])
def test_many_rows_of_each_tile(M, N, K, kind, act, tile):
    from llm_np_cp_amd.ops import hip_ops as ho

    p = ho.gemm_prompt_plan(kind, M, N, K, act, 1 << 24, 1024)
    assert (p["rows"], p["outputs"], p["parts"], p["waves"],
            p["wide"]) == tile
    test_many_rows(M, N, K, kind, act)


# tiles 256 wide by two groups of waves: slabs fewer than the ring holds, one,
# two and three, and several tiles a block (more than 256), so that one's slabs
# are asked for while another is multiplied; 256 and 128 rows, with a rest both
# ways; parts of K, also with a short last one
@pytest.mark.parametrize("M,N,K,kind,act,rows,parts", [
    (153, 11205, 12864, "bf16", -1, 128, 2),
    (223, 2589, 17600, "bf16", 0, 128, 5),
    (1025, 10942, 256, "bf16", 0, 256, 1),
    (793, 10086, 128, "fp8", -1, 256, 1), (840, 9423, 384, "fp8", -1, 256, 1),
    (332, 11127, 128, "fp8", -1, 128, 1), (330, 10970, 256, "fp8", -1, 128, 1),
    (340, 11179, 384, "fp8", -1, 128, 1),
    (195, 16680, 192, "bf16", -1, 128, 1),
    (790, 16468, 192, "bf16", -1, 128, 1),
    (1290, 10764, 320, "bf16", -1, 128, 1),
    (788, 16657, 512, "bf16", -1, 128, 1),
    (131, 16672, 768, "bf16", -1, 128, 1),
    (131, 8688, 9600, "bf16", -1, 128, 3),
    (652, 16604, 192, "bf16", -1, 256, 1),
    (1807, 13164, 192, "bf16", -1, 256, 1),
    (1409, 16516, 320, "bf16", -1, 256, 1),
    (401, 16808, 640, "bf16", -1, 256, 1),
    (196, 12624, 192, "bf16", 0, 128, 1), (341, 16438, 256, "bf16", 0, 128, 1),
    (258, 16470, 512, "bf16", 0, 128, 1), (137, 11036, 576, "bf16", 0, 128, 1),
    (130, 4100, 9600, "bf16", 0, 128, 3), (390, 14161, 128, "bf16", 0, 256, 1),
    (709, 16463, 128, "bf16", 0, 256, 1), (654, 16797, 256, "bf16", 0, 256, 1),
    (195, 16406, 576, "bf16", 0, 256, 1), (661, 16536, 576, "bf16", 0, 256, 1),
    (194, 16525, 128, "fp8", -1, 128, 1), (784, 16783, 128, "fp8", -1, 128, 1),
    (815, 16762, 512, "fp8", -1, 128, 1),
    (194, 16444, 1152, "fp8", -1, 128, 1),
    (327, 3782, 19200, "fp8", -1, 128, 4),
    (1562, 15116, 128, "fp8", -1, 256, 1),
    (1539, 15149, 512, "fp8", -1, 256, 1),
    (449, 16753, 1152, "fp8", -1, 256, 1), (261, 10856, 384, "fp8", 0, 128, 1),
    (321, 16544, 640, "fp8", 0, 128, 1), (262, 16482, 1152, "fp8", 0, 128, 1),
    (201, 2728, 12800, "fp8", 0, 128, 5), (196, 4232, 8192, "fp8", 0, 128, 3),
    (1094, 1808, 12800, "fp8", 0, 128, 3), (400, 15116, 256, "fp8", 0, 256, 1),
    (780, 15087, 384, "fp8", 0, 256, 1), (264, 13676, 896, "fp8", 0, 256, 1),
    (641, 16697, 1152, "fp8", 0, 256, 1)])
def test_many_rows_of_wide_tiles(M, N, K, kind, act, rows, parts):
    from llm_np_cp_amd.ops import hip_ops as ho

    p = ho.gemm_prompt_plan(kind, M, N, K, act, 1 << 24, 1024)
    assert p["wide"] and (p["rows"], p["parts"]) == (rows, parts)
    test_many_rows(M, N, K, kind, act)


# one row of tiles beside 32 MB of W or just less of it: read past the caches
# (once) by each tile of up to 128 rows, with a rest both ways and parts of K
@pytest.mark.parametrize("M,N,K,kind,act,tile,once", [
    (37, 8203, 2048, "bf16", 0, (64, 128, 1), True),
    (61, 2050, 8256, "bf16", -1, (64, 64, 6), True),
    (65, 16850, 1088, "bf16", -1, (128, 64, 1), True),
    (99, 9001, 2048, "bf16", -1, (64, 64, 1), False),
    (128, 14300, 2048, "bf16", 0, (128, 128, 1), True),
    (128, 28690, 640, "bf16", -1, (128, 64, 1), True),
    (128, 8190, 2048, "bf16", -1, (64, 64, 1), False),
    (70, 4110, 8192, "bf16", -1, (64, 64, 3), False),
    (33, 8203, 4096, "fp8", 0, (64, 64, 1), True),
    (57, 16500, 2176, "fp8", -1, (64, 64, 1), True),
    (128, 8400, 2176, "fp8", 0, (128, 64, 1), True),
    (121, 17010, 2112, "fp8", -1, (128, 64, 1), True),
    (128, 34000, 1024, "fp8", -1, (128, 256, 1), True),
    (128, 4099, 8320, "fp8", -1, (64, 64, 3), False),
    (67, 16613, 512, "bf16", 0, (128, 256, 1), True),
    (65, 16690, 576, "bf16", 0, (128, 256, 1), True),
    (66, 16396, 1152, "fp8", 0, (128, 256, 1), True),
    (40, 16400, 2048, "fp8", 0, (64, 128, 1), True),
    (20, 70000, 256, "bf16", -1, (32, 64, 1), True),
    (64, 8200, 4096, "bf16", -1, (64, 64, 1), True)])
def test_many_rows_beside_large_weights(M, N, K, kind, act, tile, once):
    from llm_np_cp_amd.ops import hip_ops as ho

    p = ho.gemm_prompt_plan(kind, M, N, K, act, 1 << 24, 1024)
    assert (p["rows"], p["outputs"], p["parts"]) == tile and p["once"] == once
    test_many_rows(M, N, K, kind, act)


# rows so long that 32 bits do not reach those of a tile: of the largest (256
# rows of 2^24 bytes), and of the one that takes them (64 rows of 66 MB)
@pytest.mark.parametrize("kind,act,K", [
    ("bf16", -1, (1 << 23) + 64), ("bf16", 0, (1 << 23) + 64),
    ("fp8", -1, (1 << 23) + 64), ("fp8", 0, (1 << 23) + 64),
    ("bf16", -1, 33 << 20)])
def test_long_rows(kind, act, K):
    test_many_rows(65, 70, K, kind, act)


# the tiles that the device chooses among beside MXFP4 (64x64, 64x128, 128x128
# of eight and of four waves, 128x256) with a rest both ways; fewer slabs of 64
# than buffers, as many, one more; parts of K, also with a short last one
@pytest.mark.parametrize("M,N,K", [
    (17, 70, 64), (33, 200, 8192), (64, 64, 256), (130, 1000, 320),
    (290, 900, 6144), (513, 4100, 256), (1030, 2050, 64), (1100, 2000, 4096),
    (2050, 6200, 128), (2050, 6200, 192), (2049, 3700, 1024)])
@pytest.mark.parametrize("act", [-1, 0, 1])
def test_many_rows_beside_mxfp4(M, N, K, act):
    from llm_np_cp_amd.ops import hip_ops as ho

    rows = N * (2 if act >= 0 else 1)
    W = normal(rows, K, seed=11, scale=K ** -0.5)
    X, bias, res = normal(M, K, seed=12), normal(N, seed=13), \
        normal(M, N, seed=14)
    q = torch.empty(rows, K // 2, dtype=torch.uint8, device="cuda")
    e = torch.empty(rows, K // 32, dtype=torch.uint8, device="cuda")
    ho.quant_fp4(W, q, e)
    z = X.double() @ mxfp4_values(q, e).double().T
    if act >= 0:
        f = (torch.nn.functional.silu if act == 0 else lambda t:
             torch.nn.functional.gelu(t, approximate="tanh"))
        z = f(z[:, :N]) * z[:, N:]
    part = torch.zeros(1 << 24, device="cuda")
    cnt = torch.zeros(1024, dtype=torch.int32, device="cuda")
    Y = torch.full((M + 1, N), 7.0, device="cuda").bfloat16()
    for kw, want in ((dict(), z), (dict(bias=bias, res=res, accbuf=part,
                                        cnt=cnt),
                                   z + bias.double() + res.double())):
        for _ in range(2):                          # counters are left zero
            ho.gemm_fp4w(X, q, e, Y[:M], act=act, **kw)
        # exact products, fp32 sums, bf16 results: 2^-9 at most
        assert off(Y[:M], want) < 2.0 ** -9
        assert (Y[M] == 7.0).all() and not cnt.any()


# histories of nothing, one key, a part of a tile, a block's range and one
# key more, ranges of several tiles; heads that fill no group of four; a
# window; head dims of both kernels
@pytest.mark.parametrize("hd,nh,kvh", [(16, 4, 2), (64, 3, 3), (64, 10, 2),
                                       (128, 8, 1), (256, 4, 2), (512, 2, 1)])
@pytest.mark.parametrize("pos", [0, 1, 33, 257, 1500])
@pytest.mark.parametrize("kv8", [False, True])
def test_new_tokens(hd, nh, kvh, pos, kv8):
    check_new_tokens(hd, nh, kvh, [pos, pos // 2], kv8,
                     ((1, 0, 0.0), (5, 0, 30.0), (80, 40, 0.0)))


# ranges as the device chooses them (a tile of 32 keys for each wave): more
# than the merge asks for at a time (16), as many as there may be (64 of 80),
# behind a window, and so many that the last ones get no tile (410 tiles in 45
# ranges of 10); the VALU's kernel alike
@pytest.mark.parametrize("hd,nh,kvh,at,way", [
    (64, 4, 1, [4400, 4353], (64, 0, 0.0)),
    (64, 3, 3, [16500, 700], (80, 0, 30.0)),
    (128, 8, 2, [13120, 13089], (45, 0, 0.0)),
    (128, 5, 1, [16400, 3], (80, 5000, 0.0)),
    (256, 4, 2, [2300, 8200], (64, 0, 50.0)),
    (256, 2, 1, [3000, 2177], (20, 2176, 0.0)),
    # of 256 dims: one round in one range, a key more in ranges of four
    # tiles, the last length that has those and the first that has not; where
    # the grid ends ahead of them
    (256, 4, 2, [256, 257], (64, 0, 50.0)),
    (256, 4, 2, [2048, 2049], (64, 0, 0.0)),
    (256, 8, 2, [611, 2048], (2, 0, 50.0)),
    (512, 2, 1, [1500, 1088], (80, 0, 0.0)),
    (512, 4, 2, [4500, 65], (80, 4000, 30.0)),
    (16, 4, 2, [40000, 2049], (80, 0, 0.0))])
@pytest.mark.parametrize("kv8", [False, True])
def test_new_tokens_over_many_ranges(hd, nh, kvh, at, way, kv8):
    check_new_tokens(hd, nh, kvh, at, kv8, (way,))


def check_new_tokens(hd, nh, kvh, at, kv8, ways):
    from llm_np_cp_amd.ops import hip_ops as ho

    B, S = len(at), max(at) + 9
    qkv = normal(B, (nh + 2 * kvh) * hd, seed=1)
    pools = [normal(B, kvh, S, hd, seed=2 + i) for i in range(2)]
    true, sc = [x.double() for x in pools], [None, None]
    if kv8:
        for i, x in enumerate(pools):
            q, s, t = e4m3(x.reshape(-1, hd))
            pools[i] = q.view(torch.uint8).view(x.shape).contiguous()
            sc[i], true[i] = s.view(B, kvh, S).contiguous(), t.view(x.shape)
    t = torch.arange(S, device="cuda").double()[:, None] * (
        1e4 ** -(torch.arange(hd // 2, device="cuda") * 2.0 / hd).double())
    cos, sin = t.cos().float(), t.sin().float()
    ln = torch.tensor(at, dtype=torch.int32, device="cuda")
    for split, win, cap in ways:
        part = torch.zeros(B * nh * split * (hd + 2), device="cuda")
        cnt = torch.zeros(B * nh, dtype=torch.int32, device="cuda")
        out = torch.full((B + 1, nh * hd), 7.0, device="cuda").bfloat16()
        for _ in range(2):                          # counters are left zero
            ho.attn_dec(qkv, pools[0], pools[1], out, ln, cos, sin, part, cnt,
                        nh, kvh, hd, hd ** -0.5, softcap=cap, window=win,
                        split=split, kS=sc[0], vS=sc[1], batch=B)
        for b, p in enumerate(at):
            x = qkv[b].double().view(-1, hd)
            c, s, h = cos[p].double(), sin[p].double(), hd // 2
            x[:nh + kvh] = torch.cat(
                [x[:nh + kvh, :h] * c - x[:nh + kvh, h:] * s,
                 x[:nh + kvh, h:] * c + x[:nh + kvh, :h] * s], -1)
            lo = max(0, p + 1 - win) if win else 0
            k, v = (torch.cat([true[i][b, :, lo:p],
                               x[nh + i * kvh:nh + (i + 1) * kvh, None]], 1)
                    .repeat_interleave(nh // kvh, 0) for i in range(2))
            z = (k * x[:nh, None]).sum(-1) * hd ** -0.5
            if cap:
                z = cap * torch.tanh(z / cap)
            y = (torch.softmax(z, -1)[..., None] * v).sum(1).reshape(-1)
            # fp32 all the way; the bf16 result has 8 bits: half a unit of
            # the last is at most 2^-8 of each value (2^-9 over many of them,
            # but there are as few as 64)
            assert off(out[b], y) < 2.0 ** -8
            for i in range(2):                      # the pool's new row
                row, want = pools[i][b, :, p], x[nh + i * kvh:][:kvh]
                if kv8:
                    row = row.view(torch.float8_e4m3fn).double() \
                        * sc[i][b, :, p, None].double()
                assert off(row, want) < (2.0 ** -4 if kv8 else 2.0 ** -8)
        assert (out[B] == 7.0).all() and not cnt.any()


# K: less than a load of the lanes, one and a rest, several waves with a rest,
# more loads than a wave takes, more than one pass; rows: fewer than waves,
# odd, more than a block's threads; what x may be on the way
@pytest.mark.parametrize("N,K", [(5, 64), (300, 544), (517, 3584),
                                 (33, 11008), (40, 41984), (140000, 96)])
@pytest.mark.parametrize("kind", ["bf16", "fp8", "fp4"])
@pytest.mark.parametrize("glu", [False, True])
def test_one_row(N, K, kind, glu):
    from llm_np_cp_amd.ops import hip_ops as ho

    W = normal(N * (2 if glu else 1), K, seed=4, scale=K ** -0.5)
    x, u = normal(K, seed=5), normal(K, seed=6)
    g, g2 = (normal(K, seed=s).float() for s in (7, 8))
    res, table = normal(N, seed=9), normal(3, K, seed=10)
    tok = torch.tensor([2], dtype=torch.int32, device="cuda")
    w, f, Wd = [W], ho.gemv, W.double()
    if kind == "fp8":
        q, s, Wd = e4m3(W)
        w, f = [q, s], ho.gemv_fp8
    if kind == "fp4":
        q = torch.empty(W.shape[0], K // 2, dtype=torch.uint8, device="cuda")
        e = torch.empty(W.shape[0], K // 32, dtype=torch.uint8, device="cuda")
        ho.quant_fp4(W, q, e)
        w, f, Wd = [q, e], ho.gemv_fp4, mxfp4_values(q, e)

    def rms(t):
        return t * torch.rsqrt(t.pow(2).mean() + 1e-5)

    xd, ud, hd = x.double(), u.double(), (table[2].double() * 1.5)
    h2 = (ud + rms(xd) * g.double()).bfloat16()
    hd = hd.bfloat16()
    keep = torch.full((K + 1,), 7.0, device="cuda").bfloat16()
    ways = [(dict(x=x, res=res), xd, None)]
    if kind != "bf16":
        ways.append((dict(x=x.float() * 1.001, res=res),
                     (x.float() * 1.001).double(), None))
    if K < 32768:
        ways += [
            (dict(x=x, stage=ho.STAGE_NORM, g=g, res=res),
             rms(xd) * g.double(), None),
            (dict(x=x, stage=ho.STAGE_GLU, x2=u, act=1, res=res),
             torch.nn.functional.gelu(xd, approximate="tanh") * ud, None),
            (dict(x=x, stage=ho.STAGE_NORM2, x2=u, g=g, g2=g2, res=keep),
             rms(h2.double()) * g2.double(), h2),
            (dict(x=table, stage=ho.STAGE_NORM_EMBED, x2=tok, g=g,
                  escale=1.5, res=keep), rms(hd.double()) * g.double(), hd)]
    for kw, ref, kept in ways:
        y = torch.full((N + 1,), 7.0, device="cuda")
        if glu:
            kw["act"] = 1
        f(*w, kw.pop("x"), y[:N], glu=glu, softcap=20.0, **kw)
        z = Wd @ ref
        if glu:
            z = torch.nn.functional.gelu(z[:N], approximate="tanh") * z[N:]
        z = 20.0 * torch.tanh(z / 20.0)
        if kept is None:
            z = z + res.double()
        else:       # the residual stream, rounded after fp32 sums
            assert off(keep[:K], kept.double()) < 2.0 ** -9
            assert keep[K] == 7.0
        # fp32 all the way; bf16 weights meet x rounded to bf16 (2^-8 of each
        # at most, twice through a gate), a kept row may round the other way
        assert off(y[:N], z) < (2.0 ** -7 if kind == "bf16" or kept is not None
                                else 2.0 ** -18)
        assert y[N] == 7.0


# what all threads of a block stage: a part of a trip, one, a trip and a rest,
# two, four, and one load more than that
@pytest.mark.parametrize("K", [32, 2016, 2048, 2080, 4096, 4128, 6176, 8192,
                               8224])
@pytest.mark.parametrize("kind", ["bf16", "fp8", "fp4"])
def test_one_row_of_every_staging(K, kind):
    test_one_row(37, K, kind, True)
    test_one_row(2600, K, kind, False)


# experts of a step at once: apart through the gate, added up after it
@pytest.mark.parametrize("n", [1, 2, 3, 8])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_experts_of_one_row(n, kind):
    from llm_np_cp_amd.ops import hip_ops as ho

    E, I, H = 9, 208, 144
    up, dn = (normal(E * r, k, seed=s, scale=k ** -0.5)
              for r, k, s in ((2 * I, H, 1), (H, I, 2)))
    x, res, g = normal(H, seed=3), normal(H, seed=4), normal(H, seed=5).float()
    idx = torch.randperm(E, generator=torch.Generator().manual_seed(n))[:n]
    idx = idx.int().cuda()
    p = torch.rand(n, generator=torch.Generator().manual_seed(6)).cuda()
    f, ups, dns, U, D = ho.gemv, [up], [dn], up.double(), dn.double()
    if kind == "fp8":
        (a, b, U), (c, d, D), f = e4m3(up), e4m3(dn), ho.gemv_fp8
        ups, dns = [a, b], [c, d]
    ups, dns = ([t[:r] for t in ts] for ts, r in ((ups, 2 * I), (dns, H)))
    kw, kd = (dict(sstride=s) if kind == "fp8" else {} for s in (2 * I, H))
    a = torch.full((n + 1, I), 7.0, device="cuda")
    if kind == "bf16":
        a = a.bfloat16()
    f(*ups, x, a[:n], stage=ho.STAGE_NORM, g=g, glu=True, eidx=idx,
      wstride=2 * I * H, **kw)
    y = res.clone()
    f(*dns, a[:n], y, res=y, eidx=idx, wstride=H * I, oscale=p, **kd)
    xn = x.double() * torch.rsqrt(x.double().pow(2).mean() + 1e-5) * g.double()
    z = res.double()
    for j, e in enumerate(idx.tolist()):
        t = U[e * 2 * I:(e + 1) * 2 * I] @ xn
        t = torch.nn.functional.silu(t[:I]) * t[I:]
        assert off(a[j], t) < (2.0 ** -7 if kind == "bf16" else 2.0 ** -18)
        z = z + p[j].double() * (D[e * H:(e + 1) * H] @ t)
    assert off(y, z) < 2.0 ** -7 and (a[n] == 7.0).all()


# widths: one load of a few lanes, a thread each, a rest in each number of
# loads, the widest
@pytest.mark.parametrize("H", [8, 2048, 2304, 4104, 9000, 16384])
@pytest.mark.parametrize("M", [1, 5])
def test_two_norms(M, H):
    from llm_np_cp_amd.ops import hip_ops as ho

    x, h = normal(M, H, seed=1), normal(M, H, seed=2)
    g, g2 = normal(H, seed=3).float(), normal(H, seed=4).float()
    y = torch.full((M + 1, H), 7.0, device="cuda").bfloat16()
    z = y.clone()
    y[:M] = h                                  # in place
    ho.rmsnorm(x, g, y[:M], res=y[:M], eps=1e-5, g2=g2, y2=z[:M])

    def rms(t):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-5)

    # bf16 results: 2^-8 of each value, the second from the first as it is
    assert off(y[:M], rms(x.double()) * g.double() + h.double()) < 2.0 ** -8
    ref = rms(y[:M].double()) * g2.double()
    assert off(z[:M], ref) < 2.0 ** -8
    assert (y[M] == 7.0).all() and (z[M] == 7.0).all()
    q = torch.full((M + 1, H), 5, dtype=torch.uint8, device="cuda")
    s = torch.zeros(M + 1, device="cuda")
    y[:M] = h
    ho.rmsnorm(x, g, y[:M], res=y[:M], eps=1e-5, g2=g2, q2=q, s2=s)
    got = q.view(torch.float8_e4m3fn).double() * s[:, None].double()
    # four bits: 2^-4 of each value; the scale is the largest one's
    assert off(got[:M], ref) < 2.0 ** -4
    assert torch.allclose(s[:M].double(), ref.abs().amax(1) / 448, rtol=1e-5)
    assert (q[M] == 5).all() and s[M] == 0
    ho.rmsnorm(x, g, None, q2=q, s2=s)         # the first norm, rounded once
    ref = rms(x.double()) * g.double()
    assert torch.allclose(s[:M].double(), ref.abs().amax(1) / 448, rtol=1e-6)
    want = (ref / s[:M, None].double()).float().to(torch.float8_e4m3fn)
    other = want.view(torch.uint8) != q[:M]    # fp32 sums: on the edge of two
    assert other.float().mean() < 0.001
    assert (q[M] == 5).all() and s[M] == 0


# rows of an expert: none, one, less and more than a tile of 32, 64 and 128
@pytest.mark.parametrize("M,E,top", [(1, 8, 2), (40, 8, 3), (200, 9, 2),
                                     (330, 4, 2), (70, 64, 8)])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_experts_of_many_rows(M, E, top, kind, H=192, I=320):
    from llm_np_cp_amd.ops import hip_ops as ho

    up, dn = (normal(E * r, k, seed=s, scale=k ** -0.5)
              for r, k, s in ((2 * I, H, 1), (H, I, 2)))
    x, h = normal(M, H, seed=3), normal(M, H, seed=4)
    r = torch.rand(M, E, generator=torch.Generator().manual_seed(5))
    r[:, E - 1] *= 0.01                             # hardly ever taken
    idx = r.topk(top, 1).indices.int().cuda().contiguous()
    p = torch.rand(M, top, generator=torch.Generator().manual_seed(6)).cuda()
    pairs = M * top
    order = torch.full((pairs + 3 * (pairs // 32 + E),), -1,
                       dtype=torch.int32, device="cuda")
    a = torch.full((pairs + 1, I), 7.0, device="cuda").bfloat16()
    y = torch.full((pairs + 1, H), 7.0, device="cuda").bfloat16()
    ho.expert_sort(idx, order, pairs, E)
    perm = order[:pairs].long()
    who = idx.reshape(-1).long()
    assert (perm.sort().values == torch.arange(pairs, device="cuda")).all()
    assert (who[perm].diff() >= 0).all()
    if kind == "fp8":
        (uq, us, U), (dq, ds, D), (xq, xs, X) = e4m3(up), e4m3(dn), e4m3(x)
        ho.expert_gemm(xq, uq, a[:pairs], order, pairs, E, top, H, True,
                       act=0, sx=xs, sw=us)
        aq, sa, ad = e4m3(a[:pairs])
        ho.expert_gemm(aq, dq, y[:pairs], order, pairs, E, top, I, False,
                       sx=sa, sw=ds)
    else:
        U, D, X = up.double(), dn.double(), x.double()
        ho.expert_gemm(x, up, a[:pairs], order, pairs, E, top, H, True, act=0)
        ho.expert_gemm(a[:pairs], dn, y[:pairs], order, pairs, E, top, I,
                       False)
        ad = a[:pairs].double()
    out = h.clone()
    ho.expert_sum(y, p, idx, out, M, top)
    U, D = U.view(E, 2 * I, H), D.view(E, H, I)
    za, zy = torch.zeros_like(ad), torch.zeros(pairs, H, device="cuda").double()
    for e in range(E):
        at = (who[perm] == e).nonzero()[:, 0]       # places in the order
        t = X[perm[at] // top] @ U[e].T
        if kind == "fp8":
            t = t.bfloat16().double()
        za[at] = torch.nn.functional.silu(t[:, :I]) * t[:, I:]
        zy[perm[at]] = ad[at] @ D[e].T
    # exact products, fp32 sums, bf16 results: 2^-8 of each value at most
    assert off(a[:pairs], za) < 2.0 ** -8 and off(y[:pairs], zy) < 2.0 ** -8
    z = h.double() + (y[:pairs].double().view(M, top, H)
                      * p.double()[..., None]).sum(1)
    assert off(out, z) < 2.0 ** -8 * top            # bf16 after each expert
    assert (a[pairs] == 7.0).all() and (y[pairs] == 7.0).all()


# more 128x128 tiles than CUs: outputs that end within a tile 256 wide, one
# slab, experts without rows, the first product alone past the line
@pytest.mark.parametrize("M,E,top,H,I", [
    (1500, 4, 2, 1408, 704), (1500, 4, 2, 1408, 768), (900, 64, 8, 64, 192),
    (2200, 1, 1, 2112, 1088), (520, 8, 2, 384, 1536), (300, 3, 1, 640, 5504)])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_experts_of_wide_tiles(M, E, top, H, I, kind):
    test_experts_of_many_rows(M, E, top, kind, H, I)


# more tiles than blocks: one expert's slabs are asked for while another's are
# multiplied.  Both products, the first alone; one slab, two, three, many; an
# expert with hardly a row.  The shares of experts are as above.
@pytest.mark.parametrize("M,E,top,H,I,both", [
    (1500, 4, 2, 2944, 1792, True), (1100, 8, 2, 3584, 2176, True),
    (2100, 8, 1, 128, 4224, False), (1100, 8, 2, 256, 4096, False),
    (1300, 12, 2, 384, 3328, False), (900, 3, 1, 640, 5504, False),
    (1000, 64, 8, 128, 640, False)])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_experts_of_several_tiles_a_block(M, E, top, H, I, both, kind):
    from llm_np_cp_amd.ops import hip_ops as ho

    r = torch.rand(M, E, generator=torch.Generator().manual_seed(5))
    r[:, E - 1] *= 0.01
    rows = torch.bincount(r.topk(top, 1).indices.reshape(-1), minlength=E)
    tiles = (-(-rows // 128)).sum().item()
    assert tiles * -(-2 * I // 256) > 256 + 32
    assert (tiles * -(-H // 256) > 256 + 32) == both
    assert ho.expert_gemm_plan(kind, M * top, E, I, H, 0)["wide"]
    assert ho.expert_gemm_plan(kind, M * top, E, H, I)["wide"] == both
    test_experts_of_many_rows(M, E, top, kind, H, I)


# a row, a few, a group in larger blocks, a large one in fewer; a vocabulary of
# one, one short of a block's trip, one more, several trips
@pytest.mark.parametrize("B", [1, 4, 5, 33])
@pytest.mark.parametrize("V", [1, 63, 4095, 4097, 40001, 70000])
def test_sampled_rows(B, V):
    from llm_np_cp_amd.ops import hip_ops as ho

    logits = normal(33, V, seed=11, scale=2.0)
    logits[:, V // 2] = logits[:, V // 3]           # ties: the first of them
    logits[0, V - 1] = 60.0
    i32 = dict(dtype=torch.int32, device="cuda")

    def sample(rows, greedy):
        n = len(rows)
        i64 = dict(dtype=torch.int64, device="cuda")
        ctr, gmax, pick = (torch.zeros(k, **i64) for k in (1, n, n))
        cnt, tok, at, ln = (torch.zeros(n, **i32) for _ in range(4))
        ring = torch.zeros(n, 4, **i32)
        for _ in range(2):
            ho.sample(rows, 0.05, greedy, 7, ctr, gmax, pick, tok, ring, at,
                      ln, cnt=cnt, batch=n)
        assert not gmax.any() and not pick.any() and not cnt.any()
        assert (at == 2).all() and (ln == 2).all()
        return ring[:, :2]

    got = sample(logits[:B], True)
    want = torch.from_numpy(logits[:B].float().cpu().numpy().argmax(1)).cuda()
    assert (got == want[:, None]).all()
    got = sample(logits[:B], False)
    # noise is a row's and a token's, whoever looks at it
    assert (got[:4] == sample(logits[:4], False)[:B]).all()
    x = logits[:B].float()
    kept = x.gather(1, got.long()) >= x.amax(1, keepdim=True) + math.log(0.05)
    assert kept.all() and (V < 4000 or B < 5 or len(got.unique()) > 3)


# rows that hold NaN or infinity: every choice is an expert's, others' rows are
# theirs alone
@pytest.mark.parametrize("E,top", [(4, 2), (8, 3), (64, 8)])
@pytest.mark.parametrize("bad", [math.nan, math.inf])
def test_router_of_rows_without_a_number(E, top, bad):
    from llm_np_cp_amd.ops import hip_ops as ho

    M, H = 5, 192
    h, g = normal(M, H, seed=1), torch.ones(H, device="cuda")
    wg = normal(E, H, seed=2)
    h[1, 7] = bad
    idx = torch.full((M, top), -9, dtype=torch.int32, device="cuda")
    w = torch.zeros(M, top, device="cuda")
    ho.moe_route(h, g, wg, M, top, idx, w)
    assert ((idx >= 0) & (idx < E)).all()
    assert all(len(set(r)) == top for r in idx.tolist())
    good = [0, 2, 3, 4]
    x = h[good].double()
    z = (x * torch.rsqrt(x.pow(2).mean(1, keepdim=True) + 1e-5)) @ wg.double().T
    p, i = torch.softmax(z, 1).topk(top, 1)
    assert (idx[good].long() == i).all()
    assert off(w[good], p / p.sum(1, keepdim=True)) < 2.0 ** -16


# a wave has an expert a lane: numbers that leave a butterfly of lanes short
@pytest.mark.parametrize("E", [1, 2, 3, 5, 6, 7, 9, 10, 12, 17, 33, 60, 63])
def test_router_of_any_number_of_experts(E):
    from llm_np_cp_amd.ops import hip_ops as ho

    M, H, top = 40, 192, min(3, E)
    h, g = normal(M, H, seed=1), torch.ones(H, device="cuda")
    wg = normal(E, H, seed=2)
    idx = torch.full((M, top), -9, dtype=torch.int32, device="cuda")
    w = torch.zeros(M, top, device="cuda")
    ho.moe_route(h, g, wg, M, top, idx, w)
    x = h.double()
    z = (x * torch.rsqrt(x.pow(2).mean(1, keepdim=True) + 1e-5)) @ wg.double().T
    p, i = torch.softmax(z, 1).topk(top, 1)
    assert (idx.long() == i).all()
    assert off(w, p / p.sum(1, keepdim=True)) < 2.0 ** -16


# a thread has 16 values of a head (of 24: one at a time); rows that end
# inside a block; a head's threads that are no power of two
@pytest.mark.parametrize("hd,nh,kvh", [(16, 4, 2), (24, 2, 1), (48, 3, 1),
                                       (64, 5, 1), (128, 6, 2), (256, 2, 2)])
@pytest.mark.parametrize("M,pos0", [(1, 0), (5, 901), (37, 3)])
@pytest.mark.parametrize("kv8", [False, True])
def test_rotated_rows(hd, nh, kvh, M, pos0, kv8):
    from llm_np_cp_amd.ops import hip_ops as ho

    S = pos0 + M + 1
    rows = normal(M, (nh + 2 * kvh) * hd + 8, seed=1)[:, 8:]
    x = rows.double()
    a = torch.rand(S, hd // 2, device="cuda", dtype=torch.float64) * 6
    cos, sin = torch.cos(a).float(), torch.sin(a).float()
    kind = torch.uint8 if kv8 else torch.bfloat16
    kc, vc = (torch.zeros(kvh, S, hd, device="cuda", dtype=kind)
              for _ in "kv")
    kS, vS = (torch.zeros(kvh, S, device="cuda") if kv8 else None
              for _ in "kv")
    q, k, v = rows.split([nh * hd, kvh * hd, kvh * hd], dim=1)
    ho.rope_cache(q, k, v, kc, vc, cos, sin,
                  torch.tensor([pos0], dtype=torch.int32, device="cuda"),
                  M, nh, kvh, hd, kS=kS, vS=vS)
    x = x.view(M, -1, hd)
    c, s = (t[pos0:pos0 + M, None].double() for t in (cos, sin))
    u, w = x[:, :nh + kvh].chunk(2, -1)
    turned = torch.cat([u * c - w * s, w * c + u * s], -1)
    # rounding off by half a last place: of 8 bits 2^-8 at most, e4m3's 4
    # bits 2^-4
    assert off(q.reshape(M, nh, hd), turned[:, :nh]) < 2 ** -8
    for got, sc, ref in ((kc, kS, turned[:, nh:]), (vc, vS, x[:, nh + kvh:])):
        new = got[:, pos0:pos0 + M].permute(1, 0, 2)
        if kv8:
            want = ref.abs().amax(-1) / 448
            scale = sc[:, pos0:pos0 + M].T.double()
            assert ((scale - want).abs() <= 1e-6 * want).all()
            new = new.contiguous().view(torch.float8_e4m3fn).double() * \
                scale[..., None]
            assert off(new, ref) < 2 ** -4
        else:
            assert off(new, ref) < 2 ** -8
        before = got[:, :pos0].float() if not kv8 else got[:, :pos0]
        assert not before.any() and not got[:, pos0 + M:].any()


# prompts of one batch: one wave a tile and four, a sequence that goes on
# behind earlier keys, windows, keys split over blocks, pools out of order; parts
# of the keys row by row and in lines, of which short sequences have none
@pytest.mark.parametrize("hd,nh,kvh", [(64, 8, 2), (128, 3, 1), (256, 2, 2)])
@pytest.mark.parametrize("segs,window,cap", [
    ([(0, 0, 1), (2, 0, 4)], 0, 0.0),
    ([(1, 700, 3), (0, 0, 2), (2, 31, 8)], 40, 50.0),
    ([(2, 0, 33), (0, 130, 1), (1, 0, 129)], 0, 0.0),
    ([(0, 2000, 9), (1, 0, 43), (2, 3, 300)], 64, 0.0),
    ([(2, 1500, 30), (0, 0, 12), (1, 700, 5)], 0, 0.0),
    ([(2, 2500, 40), (0, 0, 150), (1, 700, 5)], 0, 50.0)])
@pytest.mark.parametrize("kv8", [False, True])
def test_prompts_of_one_batch(hd, nh, kvh, segs, window, cap, kv8):
    from llm_np_cp_amd.ops import hip_ops as ho

    M, S = sum(n for _, _, n in segs), max(p + n for _, p, n in segs) + 3
    pool = torch.cat([torch.full((n,), b) for b, _, n in segs])
    pos = torch.cat([torch.arange(p, p + n) for _, p, n in segs])
    rows = torch.stack([pos, pool]).int().cuda()
    kc, vc = (normal(3, kvh, S, hd, seed=s) for s in (2, 3))
    kS = vS = None
    if kv8:
        (kc, kS, _), (vc, vS, _) = e4m3(kc), e4m3(vc)
    a = torch.rand(S, hd // 2, device="cuda", dtype=torch.float64) * 6
    cos, sin = torch.cos(a).float(), torch.sin(a).float()
    part = torch.zeros(1 << 22, device="cuda")
    kw = dict(softcap=cap, window=window, part=part)

    def run(x, packed):
        q, k, v = x.split([nh * hd, kvh * hd, kvh * hd], dim=1)
        caches = [t if t is None else t.clone() for t in (kc, vc, kS, vS)]
        out = torch.full((M, nh * hd), 7.0, device="cuda").bfloat16()
        if packed:
            K, V, ks, vs = caches
            ho.rope_cache(q, k, v, K, V, cos, sin, None, M, nh, kvh, hd,
                          kS=ks, vS=vs, rows=rows)
            tiles = torch.from_numpy(ho.attn_tiles(segs, nh // kvh)).cuda()
            ho.attn_prefill_mfma(
                q, K, V, out, None, M, nh, kvh, hd, hd ** -0.5, kS=ks, vS=vs,
                keys=S - 3, tiles=tiles, most=max(n for _, _, n in segs),
                **kw)
            return out, caches
        at = 0
        for b, p, n in segs:                      # each by itself
            K, V, ks, vs = (t if t is None else t[b] for t in caches)
            i = slice(at, at + n)
            p0 = torch.tensor([p], dtype=torch.int32, device="cuda")
            ho.rope_cache(q[i], k[i], v[i], K, V, cos, sin, p0, n, nh, kvh,
                          hd, kS=ks, vS=vs)
            ho.attn_prefill_mfma(q[i], K, V, out[i], p0, n, nh, kvh, hd,
                                 hd ** -0.5, kS=ks, vS=vs, keys=p + n, **kw)
            at += n
        return out, caches

    x = normal(M, (nh + 2 * kvh) * hd, seed=1, scale=2.0)
    (got, c0), (want, c1) = run(x.clone(), True), run(x.clone(), False)
    for t, u in zip(c0, c1):
        assert t is None or torch.equal(t, u)
    # keys in other ranges: sums in another order, rounded to bf16 at the end
    assert off(got, want.double()) < 2 ** -8


# row tiles of 16, outputs that end inside a tile (also where four do not fit),
# one slab, fewer slabs than waves, half a slab at the end, K split over two
# and more blocks, rows apart
@pytest.mark.parametrize("f8", [False, True])
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(16, 64), (40, 192), (4130, 320),
                                 (70, 9280), (33, 16448), (256, 4096)])
@pytest.mark.parametrize("kind", ["plain", "all", "gate"])
def test_some_rows(f8, M, N, K, kind):
    from llm_np_cp_amd.ops import hip_ops as ho

    if kind == "gate" and M > 32:
        pytest.skip("a gate takes up to 32 rows")
    act = 1 if kind == "gate" else -1
    X = normal(M, K + 32, seed=1)[:, :K]
    W = normal(N * (2 if act >= 0 else 1), K, seed=2, scale=K ** -0.5)
    Xd, Wd, kw = X.double(), W.double(), {}
    if f8:
        (X, kw["sx"], Xd), (W, kw["ws"], Wd) = e4m3(X), e4m3(W)
    ref = Xd @ Wd.T
    # fp32 sums: as many roundings as products, of the sum of magnitudes
    far = Xd.abs() @ Wd.abs().T * (K * 2.0 ** -23)
    if kind == "gate":
        g, u = ref.chunk(2, 1)
        gf, uf = far.chunk(2, 1)
        t = torch.nn.functional.gelu(g, approximate="tanh")
        # the activation's slope is at most 1.13, and 2^-20 of tanh
        far = (gf * 1.13 + g.abs() * 2.0 ** -20) * (u.abs() + uf) + \
            t.abs() * uf
        ref = t * u
    Y = torch.full((M + 1, N + 4), 7.0, device="cuda").bfloat16()
    if kind == "all":
        kw["bias"], kw["softcap"] = normal(N, seed=3), 3.0
        kw["res"] = normal(M, N + 12, seed=4)[:, :N]
        ref = 3.0 * torch.tanh(ref / 3.0) + kw["bias"].double() + \
            kw["res"].double()
        far = far + 2.0 ** -20
        Y = Y.float()
    part = torch.full((1 << 21,), float("nan"), device="cuda")
    cnt = torch.zeros(256, dtype=torch.int32, device="cuda")
    for _ in range(2):               # the counters are left zero
        ho.mid_gemm(X, W, Y[:M, :N], M, act=act, part=part, cnt=cnt, **kw)
        if f8:
            # e4m3 products are cut off at the largest one's place before
            # they are added (2^-18 of the sum seen): like more rows'
            assert off(Y[:M, :N], ref) < 2.0 ** (-9 if act < 0 else -8)
        err = (Y[:M, :N].double() - ref).abs()
        round_ = 0.0 if kind == "all" else ref.abs() * 2.0 ** -8
        assert f8 or (err <= far + round_ + 1e-30).all()
        assert (Y[M] == 7.0).all() and (Y[:, N:] == 7.0).all()
        assert not cnt.any()


# e4m3 products by instructions of 32 and of 128 values of K: both cut their
# products off at the same place, so one is as far from 64 bits as the other
@pytest.mark.parametrize("M,K", [(2, 512), (9, 2048), (16, 8192)])
@pytest.mark.parametrize("kind", ["normal", "outliers", "cubes", "positive"])
def test_e4m3_sums_of_both_instructions(M, K, kind):
    from llm_np_cp_amd.ops import hip_ops as ho

    N = 16384                        # row_gemm does not hand it on
    X = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).cuda()
    W = torch.randn(N, K, generator=torch.Generator().manual_seed(K)).cuda()
    if kind == "outliers":
        X[:, ::97] *= 30
    elif kind == "cubes":
        X, W = X ** 3, W ** 3
    elif kind == "positive":
        X, W = X.abs(), W.abs()
    (x, sx, Xd), (w, ws, Wd) = e4m3(X), e4m3(W)
    ref, far = Xd @ Wd.T, []
    for f in (ho.row_gemm, ho.mid_gemm):
        Y = torch.empty(M, N, device="cuda")
        f(x, w, Y, M, ws=ws, sx=sx)
        far.append(off(Y, ref))
    assert far[0] < 2.0 ** -13           # 6e-5 seen, of cubes
    assert far[1] <= far[0] * 1.01


# counters are the caller's or the call's own
def test_mxfp4_products_without_counters():
    from llm_np_cp_amd.ops import hip_ops as ho

    M, N, K = 33, 200, 8192
    W, X = normal(N, K, seed=1, scale=K ** -0.5), normal(M, K, seed=2)
    q = torch.empty(N, K // 2, dtype=torch.uint8, device="cuda")
    e = torch.empty(N, K // 32, dtype=torch.uint8, device="cuda")
    ho.quant_fp4(W, q, e)
    part = torch.full((1 << 22,), float("nan"), device="cuda")
    cnt = torch.zeros(1024, dtype=torch.int32, device="cuda")
    a, b = (torch.empty(M, N, device="cuda").bfloat16() for _ in "ab")
    ho.gemm_fp4w(X, q, e, a, accbuf=part, cnt=cnt)
    assert not part[0].isnan()                   # K is split
    part.fill_(float("nan"))
    ho.gemm_fp4w(X, q, e, b, accbuf=part)
    assert not part[0].isnan() and torch.equal(a, b)
