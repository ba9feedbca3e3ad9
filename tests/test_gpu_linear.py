"""Staged rows of the layer-list kernels, within and beyond the registers."""

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
