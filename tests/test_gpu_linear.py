"""Products and staged rows of the layer-list kernels at the sizes where their
launches change: tiles and buffers of the row products, few rows with fewer
slabs than waves, rows within and beyond the registers, experts by rows a
tile."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "fp32": torch.float32}
# relative rounding of a result kept in the type: half a step of 8 (24) bits
ROUND = {"bf16": 2.0 ** -8, "fp32": 2.0 ** -24}


@pytest.fixture(scope="module")
def hy():
    from llm_np_cp_amd.ops import hybrid_ops
    return hybrid_ops


def draw(seed, *shape, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(dtype).cuda()


# A sum of K products in fp32 is off by at most K roundings of the sum of
# their magnitudes (2^-24 each, twice that where a unit truncates).
def product(X, W):
    x, w = X.double(), W.double()
    return x @ w.T, x.abs() @ w.abs().T * (X.shape[1] * 2.0 ** -23)


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("M,N", [
    (65, 70), (100, 2050),        # 64x64, few tiles
    (1100, 1990), (1100, 2500),   # 64x64, more than two a CU
    (1100, 2800),                 # 128x64
    (1100, 4090),                 # 128x64, more than two a CU
    (1100, 5100),                 # 128x128
])
@pytest.mark.parametrize("K", [64, 192, 576])
def test_tiles_of_row_products(hy, dtype, M, N, K):
    X, W = draw(M, M, K, dtype=DT[dtype]), draw(N, N, K, dtype=DT[dtype])
    Y = torch.full((M + 1, N), 7.0, device="cuda")
    hy.gemm_rows(X, W, Y, M, K, N, hy.EPI_F32)
    want, far = product(X, W)
    assert ((Y[:M].double() - want).abs() <= far).all()
    assert (Y[M] == 7.0).all()


# blocks of 8, 16 and 32 outputs by 8 and 16 waves, with a rest of outputs and
# of slabs: the first and last numbers of blocks of 16, and of slabs, of each
@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("M", [2, 8, 9, 16])
@pytest.mark.parametrize("N,slabs", [
    (40, 16), (2044, 19), (2050, 16), (3058, 32), (4092, 33), (4100, 16),
    (6140, 70), (6150, 16), (6150, 64), (8190, 63), (8200, 31), (8200, 32),
    (8200, 129), (16372, 33), (16390, 32), (16390, 31)])
def test_few_rows_by_blocks(hy, dtype, M, N, slabs):
    K = slabs * (64 if dtype == "bf16" else 32)
    K += K % 64                          # rows are padded to 64
    X, W = draw(M, M, K, dtype=DT[dtype]), draw(N, N, K, dtype=DT[dtype])
    b = draw(3, N, dtype=torch.float32)
    Y = torch.full((M + 1, N), 7.0, device="cuda")
    hy.gemm_rows(X, W, Y, M, K, N, hy.EPI_F32, bias=b)
    want, far = product(X, W)
    want = want + b.double()
    assert ((Y[:M].double() - want).abs() <= far + want.abs() * 2.0 ** -23).all()
    assert (Y[M] == 7.0).all()


# pairs of columns that turn in each kind of block
@pytest.mark.parametrize("N", [264, 2584, 4168, 8264])
def test_few_rows_turned(hy, N):
    M, K, RT, dims, split = 5, 2048, 8, 6, N - 64
    X, W = (draw(k, n, K, dtype=DT["bf16"]) for k, n in ((1, M), (2, N)))
    ang = torch.rand(40, dims // 2, device="cuda", dtype=torch.float64) * 6
    pos = torch.arange(7, 7 + M, dtype=torch.int32, device="cuda")
    cos, sin = torch.cos(ang).float(), torch.sin(ang).float()
    Y = torch.full((M + 1, N), 7.0, device="cuda").bfloat16()
    R = torch.full((M + 1, 8, 16), 7.0, device="cuda").bfloat16()
    rot = hy.Rotary().put(pos=pos, cosT=cos, sinT=sin, y=R, split=split,
                          RT=RT, dims=dims, ld=128, hs=16)
    hy.gemm_rows(X, W, Y, M, K, N, hy.EPI_ROTARY, rotary=rot)
    want, far = product(X, W)
    t = want[:, split:].view(M, 8, RT).clone()
    c, s = (f[pos.long(), None].double() for f in (cos, sin))
    a, b = t[..., :dims:2].clone(), t[..., 1:dims:2].clone()
    t[..., :dims:2], t[..., 1:dims:2] = a * c - b * s, b * c + a * s
    # rounded to bf16 at the end; a turn adds up two products
    for got, w, f in ((Y[:M, :split], want[:, :split], far[:, :split]),
                      (R[:M, :, :RT], t, 2 * far[:, split:].view(M, 8, RT)
                       .amax(-1, keepdim=True) + t.abs() * 2.0 ** -22)):
        assert ((got.double() - w).abs() <= f + w.abs() * 2.0 ** -8).all()
    assert (Y[:, split:] == 7.0).all() and (R[..., RT:] == 7.0).all()
    assert (Y[M] == 7.0).all() and (R[M] == 7.0).all()


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("M", [2, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(72, 64), (528, 512), (2056, 1088)])
def test_few_rows_of_few_slabs(hy, dtype, M, N, K):
    X, W = draw(M, M, K, dtype=DT[dtype]), draw(N, N, K, dtype=DT[dtype])
    Y = torch.full((M + 1, N), 7.0, device="cuda")
    hy.gemm_rows(X, W, Y, M, K, N, hy.EPI_F32)
    want, far = product(X, W)
    assert ((Y[:M].double() - want).abs() <= far).all()
    assert (Y[M] == 7.0).all()


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("W", [60, 2048, 2052, 4096, 4100, 6144])
@pytest.mark.parametrize("form", ["norm", "gate", "xadd", "both", "sum"])
def test_staged_rows(hy, dtype, W, form):
    M, Kp, eps = 3, -(-W // 64) * 64, 1e-5
    x, y, xadd = (draw(i, M, W) for i in range(3))
    g, gb = draw(3, W), draw(4, W)
    gate = draw(5, M, W + 4)
    out = torch.full((M + 1, Kp), 7.0, device="cuda", dtype=DT[dtype])
    xout = torch.zeros(M, W, device="cuda")
    kw = {}
    v, size = x.double(), x.double().abs()
    if form == "sum":
        kw.update(y=y, gb=gb)
        t = y.double()
        t = t / (t * t).mean(-1, keepdim=True).add(eps).sqrt() * gb.double()
        v, size = v + t, size + t.abs()
    if form in ("xadd", "both", "sum"):
        kw.update(xadd=xadd, xout=xout)
        v, size = v + xadd.double(), size + xadd.double().abs()
    by = g.double() / (v * v).mean(-1, keepdim=True).add(eps).sqrt()
    if form in ("gate", "both"):
        kw.update(gate=gate, ldg=W + 4)
        by = by * torch.sigmoid(gate[:, :W].double())
    hy.norm_rows(x, g, out, M, W, Kp, eps, **kw)
    # a thread adds up to W/256 squares, a tree of 8 follows: 33 roundings,
    # halved by the root, of each of two norms, and a dozen of the products
    far = 2.0 ** -18
    want = v * by
    assert ((out[:M, :W].double() - want).abs()
            <= far * size * by.abs() + ROUND[dtype] * want.abs()).all()
    assert (out[:M, W:] == 0).all() and (out[M] == 7.0).all()
    if "xout" in kw:
        assert ((xout.double() - v).abs() <= far * size).all()


# the last number of short rows that eight waves take each, and the first that
# four do
@pytest.mark.parametrize("M", [512, 513])
@pytest.mark.parametrize("W", [1030, 2048])
@pytest.mark.parametrize("form", ["norm", "gate", "sum"])
def test_many_staged_rows(hy, M, W, form):
    Kp, eps = -(-W // 64) * 64, 1e-5
    x, y, gate = (draw(i, M, W) for i in range(3))
    g, gb = draw(3, W), draw(4, W)
    out = torch.full((M + 1, Kp), 7.0, device="cuda")
    v, size, kw = x.double(), x.double().abs(), {}
    if form == "sum":
        kw.update(y=y, gb=gb, xout=x)                 # in its place
        t = y.double()
        t = t / (t * t).mean(-1, keepdim=True).add(eps).sqrt() * gb.double()
        v, size = v + t, size + t.abs()
    by = g.double() / (v * v).mean(-1, keepdim=True).add(eps).sqrt()
    if form == "gate":
        kw.update(gate=gate, ldg=W)
        by = by * torch.sigmoid(gate.double())
    hy.norm_rows(x, g, out, M, W, Kp, eps, **kw)
    far = 2.0 ** -18                    # as for few rows
    assert ((out[:M, :W].double() - v * by).abs()
            <= far * size * by.abs()).all()
    assert (out[:M, W:] == 0).all() and (out[M] == 7.0).all()
    assert ((x.double() - v).abs() <= far * size).all()


@pytest.mark.parametrize("dtype", ["bf16", "fp32"])
@pytest.mark.parametrize("T,bm", [
    (5, 32), (90, 32), (150, 64),
    (700, 64),                    # more blocks than two a CU
    (700, 128)])
def test_experts_by_rows_a_tile(hy, dtype, T, bm):
    E, top, W, ff = 4, 2, 1088, 1024
    dt = DT[dtype]
    gu = draw(0, E, 2 * ff, W, dtype=dt) * W ** -0.5
    down = draw(1, E, W, ff, dtype=dt) * ff ** -0.5
    h = draw(2, T, W, dtype=dt)
    gen = torch.Generator().manual_seed(T)
    idx = torch.stack([torch.randperm(E, generator=gen)[:top]
                       for _ in range(T)]).int().cuda()
    wt = torch.rand(T, top, generator=gen).cuda()
    pairs, tiles = T * top, T * top // bm + E
    i32 = dict(device="cuda", dtype=torch.int32)
    perm = torch.zeros(pairs, **i32)
    at = [torch.zeros(tiles, **i32) for _ in range(3)]
    act = torch.zeros(pairs, ff, device="cuda", dtype=dt)
    y = torch.zeros(pairs, W, device="cuda", dtype=dt)
    x = torch.full((T, W), 7.0, device="cuda")
    m = hy.MoeArgs().put(h=h, gu=gu, down=down, idx=idx, wt=wt, act=act,
                         ldh=W, ldact=ff, W=W, E=E, K1=top, ff=ff, ffs=0,
                         glu=1, win=0, lim=0.0, lims=0.0)
    s = hy.MoeSort().put(perm=perm, tile_e=at[0], tile_row0=at[1],
                         tile_n=at[2], pairs=pairs, groups=E, bm=bm,
                         maxtiles=tiles)
    hy.moe_rows(int(dt == torch.float32), m, s, y, x, T, 1.0, True)
    want = torch.zeros(T, W, device="cuda", dtype=torch.float64)
    far = torch.zeros_like(want)
    r = ROUND[dtype]
    for e in range(E):
        # 16 gate rows, then their 16 up rows
        rows = gu[e].view(ff // 16, 2, 16, W)
        g, dg = product(h, rows[:, 0].reshape(ff, W))
        u, du = product(h, rows[:, 1].reshape(ff, W))
        a = torch.nn.functional.silu(g) * u
        # the slope of silu stays below 1.1; its own rounding is in 2^-20
        da = (1.1 * dg * (u.abs() + du) + (g.abs() + dg) * du
              + (r + 2.0 ** -20) * a.abs())
        d = down[e].double()
        o = a @ d.T
        do = da @ d.abs().T + a.abs() @ d.abs().T * (ff * 2.0 ** -23)
        do = do + r * (o.abs() + do)
        by = ((idx == e) * wt).sum(1, keepdim=True).double()
        want += by * o
        far += by * (do + 2.0 ** -21 * o.abs())
    assert ((x.double() - want).abs() <= far).all()
