"""How few-row products are laid out, by host arithmetic: whatever the room
for their parts, every size is taken and stays within it."""

import pytest

from llm_np_cp_amd.core.config import PRESETS, preset_config
from llm_np_cp_amd.ops import hip_ops as ho

LDS = 160 * 1024 - 1024          # of a block, less what is declared statically


@pytest.fixture(scope="module", autouse=True)
def built():
    from csrc.build import ensure_built
    ensure_built(names=["llmops"])


def cdiv(a, b):
    return -(-a // b)


def check(kind, M, N, K, glu, norm, part, cnt=256):
    p = ho.row_gemm_plan(kind, M, N, K, glu, norm, part, cnt)
    assert p is not None
    P, slab = 2 if glu else 1, {"bf16": 64, "fp8": 128, "fp4": 256}[kind]
    tiles, ks = cdiv(p["outputs"], p["tile"]), p["splits"]
    assert 1 <= p["rows"] <= M
    # every part of K has a slab, every block an output
    assert p["k"] % slab == 0 and (ks - 1) * p["k"] < K <= ks * p["k"]
    assert (p["blocks"] - 1) * p["outputs"] < N <= p["blocks"] * p["outputs"]
    # rows of X and what eight waves have of the tiles
    x = p["rows"] * (p["k"] * (1 if kind == "fp8" else 2) + 16)
    assert x + (tiles + 7) * P * 1024 == p["lds"] <= LDS
    if ks > 1:
        assert not norm and p["blocks"] <= cnt
        assert p["blocks"] * tiles * ks * P * 256 == p["floats"] <= part
    return p


def products(c):
    H, I, hd = c.hidden_size, c.intermediate_size, c.head_dim
    nh, kvh = c.num_attention_heads, c.num_key_value_heads
    return [((nh + 2 * kvh) * hd, H, False), (H, nh * hd, False),
            (I, H, True), (H, I, False), (c.vocab_size, H, False)]


@pytest.mark.parametrize("name", sorted(PRESETS))
@pytest.mark.parametrize("kind", ["bf16", "fp8", "fp4"])
def test_every_preset_at_any_room(name, kind):
    c = preset_config(name)
    for N, K, glu in products(c):
        if K % 64:
            continue
        for M in range(1, ho.FEW_ROWS + 1):
            for rows in (0, 1, 16, 64, 256, 2048):
                part = rows * max(c.hidden_size, c.intermediate_size)
                check(kind, M, N, K, glu, False, part)
                if K <= ho.ROW_NORM_K:
                    check(kind, M, N, K, glu, True, part)
        room = ho.row_gemm_room(kind, N, K, glu)
        for M in range(1, ho.FEW_ROWS + 1):     # as much as is asked for
            assert check(kind, M, N, K, glu, False, room)["rows"] == M


# sums that just do and just do not fit beside X; parts that end up with no
# slab (13 of 16); more column groups than counters
@pytest.mark.parametrize("kind,M,N,K", [
    ("bf16", 8, 4608, 9536), ("fp4", 5, 4104, 14208), ("bf16", 3, 4104, 25536),
    ("fp4", 1, 100, 26944), ("bf16", 16, 152064, 5120),
    ("bf16", 16, 128256, 8192), ("fp8", 16, 30000, 28672)])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("part", [0, 1 << 16, 1 << 20, 1 << 40])
@pytest.mark.parametrize("cnt", [16, 256])
def test_edges_of_room(kind, M, N, K, glu, part, cnt):
    p = check(kind, M, N, K, glu, False, part, cnt)
    if part == 0:
        assert p["splits"] == 1


def test_refused():
    assert ho.row_gemm_plan("bf16", 17, 64, 64) is None
    assert ho.row_gemm_plan("bf16", 1, 64, 96) is None
    assert ho.row_gemm_plan("bf16", 1, 64, 1 << 17, part=0) is None
    assert ho.row_gemm_plan("bf16", 1, 64, 1 << 17) is not None
