"""What products of many rows run by, on the host alone: the tiles that were
measured to be far from the best are not chosen."""

import pytest

from llm_np_cp_amd.ops import hip_ops as ho


@pytest.fixture(scope="module", autouse=True)
def built():
    from csrc.build import ensure_built
    ensure_built(names=["llmops"])


def plan(kind, M, N, K, act=-1):
    return ho.gemm_prompt_plan(kind, M, N, K, act, part=2048 * 14336)


# e4m3 rows that end with half a slab do not go by the two groups of waves, and
# are not to be priced as if they did: 128x256 by one group took up to 1.5 times
# as long as smaller tiles
@pytest.mark.parametrize("M,N,K", [
    (2000, 5120, 1728), (611, 14336, 1728), (611, 14336, 2368),
    (1500, 7168, 4544), (1792, 4786, 704), (1115, 9382, 576)])
def test_half_a_slab_is_not_priced_as_whole_ones(M, N, K):
    assert plan("fp8", M, N, K)["outputs"] < 256


@pytest.mark.parametrize("M,N,K,act", [
    (2048, 28672, 4096, -1), (2048, 14336, 4096, 0), (1999, 6144, 4096, -1),
    (611, 14336, 3584, 0)])
def test_only_whole_slabs_go_by_two_groups_of_waves(M, N, K, act):
    assert plan("fp8", M, N, K, act)["wide"]
    assert not plan("fp8", M, N, K + 64, act)["wide"]
    assert plan("bf16", M, N, K, act)["wide"]
    assert not plan("fp4", M, N, K, act)["wide"]


# few slabs: what a tile takes before its first product and behind its last
# weighs more than a slab, by 128x128 tiles of four waves above all
@pytest.mark.parametrize("kind,M,N,K,act", [
    ("bf16", 789, 1536, 576, 0), ("bf16", 1159, 1536, 576, 0),
    ("bf16", 746, 1748, 768, 0), ("bf16", 1883, 1152, 896, -1),
    ("bf16", 1024, 2344, 384, -1), ("bf16", 226, 10756, 832, -1)])
def test_few_slabs_are_not_for_four_waves(kind, M, N, K, act):
    assert plan(kind, M, N, K, act)["waves"] == 8


# outputs that are no multiple of four leave one by one: a large tile has most
@pytest.mark.parametrize("M,N,K", [(144, 16890, 384), (397, 8358, 512),
                                   (388, 8605, 832), (816, 4690, 128)])
def test_outputs_that_leave_one_by_one(M, N, K):
    p = plan("bf16", M, N, K)
    assert p["rows"] * p["outputs"] < 128 * 128


# no more row tiles are counted on than experts of as many rows each have: those
# leave small tiles one a CU, which end before half as many wide ones
@pytest.mark.parametrize("M,E,top,N,K,act,wide", [
    (848, 8, 2, 2048, 4096, -1, False), (456, 4, 2, 4096, 14336, -1, False),
    (192, 4, 4, 2048, 4096, 0, False), (1100, 8, 2, 2048, 4096, -1, True),
    (1100, 8, 2, 4096, 2048, 0, True), (700, 8, 2, 14336, 4096, 0, True),
    (700, 8, 2, 2048, 4096, -1, False), (300, 8, 2, 14336, 4096, 0, False)])
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_wide_tiles_of_experts(M, E, top, N, K, act, wide, kind):
    p = ho.expert_gemm_plan(kind, M * top, E, N, K, act)
    assert p["wide"] == wide and (p["rows"] == 128 or not wide)
    if kind == "fp8":
        assert not ho.expert_gemm_plan(kind, M * top, E, N, K + 64, act)["wide"]
