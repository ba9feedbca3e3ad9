"""How prompt attention goes about a call, by host arithmetic: what its blocks
are given to do where another way was measured to take longer."""

import pytest

from llm_np_cp_amd.ops import hip_ops as ho


@pytest.fixture(scope="module", autouse=True)
def built():
    from csrc.build import ensure_built
    ensure_built(names=["llmops"])


def plan(hd, nh, kvh, segs, window=0, kv8=False, part=1 << 24):
    """Of one sequence (position, rows) or of several packed ones."""
    M, most = sum(n for _, n in segs), max(n for _, n in segs)
    kw = {}
    if len(segs) > 1:
        tiles = ho.attn_tiles([(i, *s) for i, s in enumerate(segs)], nh // kvh)
        kw = dict(most=most, ntiles=len(tiles))
    return ho.attn_prefill_plan(M, nh, kvh, hd, max(p + n for p, n in segs),
                                window, kv8, part, **kw)


# Some twenty rows behind thousands of keys: dozens of parts of each, which a
# block of 16 rows would add one after the other (15 us, so 20); from a part of
# 128 rows on, and of few parts, such blocks are the better ones.
@pytest.mark.parametrize("hd,nh,kvh,M,pos0,by_row", [
    (64, 9, 3, 21, 7486, True), (64, 14, 2, 14, 7746, True),
    (128, 28, 4, 11, 7167, True), (256, 16, 8, 55, 4644, True),
    (256, 4, 1, 150, 900, True), (64, 32, 8, 300, 4000, False),
    (64, 16, 4, 40, 290, False), (128, 16, 4, 400, 600, False),
    (256, 16, 8, 120, 400, False)])
def test_parts_of_few_rows_lie_row_by_row(hd, nh, kvh, M, pos0, by_row):
    p = plan(hd, nh, kvh, [(pos0, M)])
    rows = M * nh
    assert p["ranges"] > 1 and not p["two"]
    assert p["by_row"] == by_row == (p["ranges"] >= 8 and
                                     rows < 128 * p["ranges"])


def test_one_wave_of_rows_lies_row_by_row():
    p = plan(64, 32, 8, [(300, 5)])
    assert p["ranges"] > 1 and p["by_row"]
    assert plan(64, 32, 8, [(300, 5)], part=0)["ranges"] == 1
