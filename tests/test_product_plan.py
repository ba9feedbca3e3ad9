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
