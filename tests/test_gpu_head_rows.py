"""The head of several rows beside e4m3 weights against 64 bits, and as exact
as a row alone."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ho():
    from llm_np_cp_amd.ops import hip_ops
    return hip_ops


def rand(seed, *shape):
    g = torch.Generator("cuda").manual_seed(seed)
    return torch.randn(*shape, generator=g, device="cuda")


# one slab and less than one a wave, a rest of slabs, tiles and blocks that end
@pytest.mark.parametrize("M", [1, 2, 7, 16])
@pytest.mark.parametrize("N,K", [(1, 64), (17, 128), (64, 320), (1000, 576),
                                 (513, 2304), (4100, 3584)])
@pytest.mark.parametrize("cap", [0.0, 30.0])
def test_head_rows(ho, M, N, K, cap):
    """Normed values in 24 bits (three of 8) and exact products: what sums in
    32 bits and the norm's factor are off."""
    x = (3 * rand(M, 40, K)).bfloat16()
    g = 1 + 0.1 * rand(2, K)
    w = (rand(3, N, K) * K ** -0.5).bfloat16()
    q = torch.empty(N, K, dtype=torch.uint8, device="cuda")
    s = torch.empty(N, device="cuda")
    ho.quant_fp8(w, q, s)
    rows = (torch.arange(M, dtype=torch.int32, device="cuda") * 7 + 3) % 40
    parts = torch.full((3 * ho.HEAD_ROWS * K,), float("nan"), device="cuda",
                       dtype=torch.bfloat16)
    y = torch.full((M + 1, N), 7.0, device="cuda")
    ho.head_rows(x, rows, q, s, y, M, g, parts, eps=1e-5, softcap=cap)
    xd = x[rows.long()].double()
    xn = xd / torch.sqrt((xd * xd).mean(1, keepdim=True) + 1e-5) * g.double()
    W = q.view(torch.float8_e4m3fn).double() * s.double()[:, None]
    z, far = xn @ W.T, xn.abs() @ W.abs().T * (K * 2.0 ** -24 + 2.0 ** -20)
    if cap:
        z, far = cap * torch.tanh(z / cap), far + cap * 2.0 ** -20
    err = (y[:M].double() - z).abs()
    assert (err <= far + 1e-30).all()
    assert (y[M] == 7.0).all()
    one = torch.empty(N, device="cuda")
    alone = 0.0
    for i in range(M):
        ho.gemv_fp8(q, s, x[rows[i]], one, stage=ho.STAGE_NORM, g=g, eps=1e-5,
                    softcap=cap)
        alone = max(alone, (one.double() - z[i]).norm().item())
    # no further off than a row alone, but for the order of a few sums
    assert err.norm(dim=1).max() <= 2 * alone + 1e-6 * z.norm(dim=1).max()


def test_refused(ho):
    x = torch.zeros(2, 96, dtype=torch.bfloat16, device="cuda")
    a = dict(rows=torch.zeros(20, dtype=torch.int32, device="cuda"),
             g=torch.ones(128, device="cuda"),
             parts=torch.zeros(1 << 14, dtype=torch.bfloat16, device="cuda"))
    for K, M in ((96, 2), (128, 0), (128, 17)):
        x = torch.zeros(20, K, dtype=torch.bfloat16, device="cuda")
        with pytest.raises(RuntimeError):
            ho.head_rows(x, Wq=torch.zeros(32, K, dtype=torch.uint8,
                                           device="cuda"),
                         scales=torch.ones(32, device="cuda"),
                         y=torch.zeros(20, 32, device="cuda"), M=M, **a)
