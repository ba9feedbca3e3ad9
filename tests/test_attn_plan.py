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


# Two groups of waves a block wait for each other and meet at the end: not worth
# it for a few tiles, which several short sequences have, however many blocks
# they are, nor where the longest block is hardly longer than the others.
@pytest.mark.parametrize("hd,nh,kvh,segs,window,kv8", [
    (64, 128, 8, [(0, 300)], 0, False),                 # five tiles
    (64, 64, 64, [(0, 600)], 100, False),               # three in a window
    (64, 40, 8, [(0, 50)] * 7 + [(1500, 30)], 0, False),
    (64, 16, 4, [(0, 199), (2849, 484), (0, 572)], 0, False),
    (128, 40, 40, [(0, 50)] * 8, 0, False),
    (128, 40, 40, [(0, 50)] * 8, 152, True),
    (128, 28, 4, [(0, 333)] * 6, 0, False),
    (128, 64, 8, [(0, 376)], 40, False),
    (128, 8, 1, [(0, 1066)], 0, False),
    (128, 32, 8, [(2000, 1999)], 0, False)])
def test_one_group_of_waves(hd, nh, kvh, segs, window, kv8):
    assert not plan(hd, nh, kvh, segs, window, kv8)["two"]


# and where a chain half as long is
@pytest.mark.parametrize("hd,nh,kvh,segs,window,kv8", [
    (64, 32, 8, [(0, 611)], 0, False), (64, 32, 8, [(0, 1999)], 0, False),
    (64, 32, 8, [(1300, 700)], 0, False), (64, 32, 8, [(300, 500)], 200, False),
    (64, 32, 8, [(0, 400), (60, 480), (0, 20)], 0, False),
    (128, 32, 8, [(0, 1000)], 0, False), (128, 24, 8, [(0, 1999)], 0, False),
    (128, 24, 8, [(0, 1999)], 0, True), (128, 32, 8, [(100, 480)], 130, False),
    (128, 64, 8, [(0, 750), (0, 101)], 0, False),
    (128, 32, 8, [(0, 400), (60, 480), (0, 20)], 0, True)])
def test_two_groups_of_waves(hd, nh, kvh, segs, window, kv8):
    assert plan(hd, nh, kvh, segs, window, kv8)["two"]


def test_two_groups_of_waves_have_two_halves_at_most():
    assert not plan(256, 16, 8, [(0, 1999)])["two"]
    assert not plan(64, 32, 8, [(0, 1999)], kv8=True)["two"]
    assert not plan(64, 32, 8, [(0, 2048)] * 2)["two"]    # 1024 blocks


# what the launch refuses the plan refuses too: no rows, no heads, heads that are
# no multiple of the kv heads, several sequences without their longest (these
# counts are divided by, on the host), another head dim
REFUSED = [dict(M=0), dict(nh=0), dict(nh=-4), dict(kvh=0), dict(kvh=-2),
           dict(nh=5), dict(ntiles=3), dict(ntiles=-1, most=2), dict(hd=96)]


@pytest.mark.parametrize("bad", REFUSED)
def test_plan_refuses_what_the_launch_does(bad):
    kw = dict(M=4, nh=4, kvh=2, hd=64, keys=100, part=1 << 20)
    assert ho.attn_prefill_plan(**kw)["ranges"] > 0
    with pytest.raises(RuntimeError):
        ho.attn_prefill_plan(**{**kw, **bad})


# refused by its counts, before any pointer or the device is looked at
@pytest.mark.parametrize("bad", REFUSED)
def test_launch_refuses_bad_counts(bad):
    c = dict(dict(M=4, nh=4, kvh=2, hd=64, most=0, ntiles=0), **bad)
    at = 1 << 12                       # there or not is all that is asked
    rc = ho.lib().launch_attn_prefill_mfma(
        0, 0, 0, 0, 0, at if c["ntiles"] else 0, 0, 0, at, 1 << 20, 0, c["M"],
        c["nh"], c["kvh"], c["hd"], 512, 128, 100, c["most"], c["ntiles"], 0.1,
        0.0, 0, 0)
    assert rc == 1                     # hipErrorInvalidValue
