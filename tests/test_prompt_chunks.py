"""Which rows of a group's prompts share a chunk, and their tiles."""

import types

import numpy as np
import pytest

from llm_np_cp_amd.models.engine import GPUModel
from llm_np_cp_amd.ops import hip_ops as ho


def chunks(lens, PC=64, fp8=False, wq4=False, hd=64, rows=None):
    m = types.SimpleNamespace(PC=PC, fp8=fp8, wq4=wq4, hd=hd)
    return GPUModel._chunks(m, lens, rows)


@pytest.mark.parametrize("kind", [{}, {"fp8": True},
                                  {"fp8": True, "wq4": True}, {"hd": 80}])
@pytest.mark.parametrize("lens", [[1], [64, 64], [5, 40, 1, 33, 64, 2],
                                  [200, 3, 65, 129], [1, 1, 1]])
def test_every_row_once_in_order(lens, kind):
    out = chunks(lens, **kind)
    assert all(0 < sum(n for _, _, n in c) <= 64 for c in out)
    seen = {}
    for c in out:
        for b, p, n in c:
            assert n > 0 and p == seen.get(b, 0)
            seen[b] = p + n
    assert [seen[b] for b in range(len(lens))] == lens
    if "hd" in kind:
        assert all(len(c) == 1 for c in out)
    if lens == [1, 1, 1] and kind != {"fp8": True} and "hd" not in kind:
        assert len(out) == 1
    for c in out:                  # as ever: one row beside e4m3 by itself
        if kind == {"fp8": True} and len(c) > 1:
            assert all(lens[b] % 64 != 1 for b, _, _ in c)


# a row beside e4m3 weights is in a chunk by itself, and so not rounded, where
# it is when its prompt is read alone, and nowhere else
@pytest.mark.parametrize("PC", [1, 2, 3, 4, 5, 64])
def test_a_row_by_itself_whatever_its_neighbours(PC):
    rng = np.random.default_rng(PC)
    lists = [[40, 25], [63, 2], [63, 3], [2, 63], [62, 2, 2], [64, 65, 66]]
    lists += [rng.integers(1, 3 * PC + 4, size=rng.integers(1, 9)).tolist()
              for _ in range(500)]
    for lens in lists:
        out, seen = chunks(lens, PC=PC, fp8=True), [0] * len(lens)
        single = [c[0][:2] for c in out if sum(n for _, _, n in c) == 1]
        for c in out:
            assert 0 < sum(n for _, _, n in c) <= PC
            for b, p, n in c:
                assert n > 0 and p == seen[b]
                seen[b] += n
        assert seen == lens
        assert single == [(b, p) for b, n in enumerate(lens)
                          for p in range(0, n, PC) if n - p == 1 or PC == 1]


def test_a_long_prompt_with_chunks_of_its_own():
    """In the chunks that it is read in without a group."""
    def rows(n):
        return 64 if n <= 64 else 48

    def cut(b, n, most):
        return [[(b, p, min(most, n - p))] for p in range(0, n, most)]

    for n in (1, 64, 65, 100, 200):
        assert chunks([n], rows=rows) == cut(0, n, rows(n))
        assert chunks([n, 70], hd=80, rows=rows) == \
            cut(0, n, rows(n)) + cut(1, 70, 48)
        assert chunks([n, 70], rows=rows) == chunks([n, 70])


@pytest.mark.parametrize("group", [1, 3, 7])
@pytest.mark.parametrize("segs", [
    [(0, 0, 1)], [(3, 7, 4), (1, 0, 2)], [(0, 0, 200), (2, 900, 33)],
    [(1, 0, 43), (0, 5, 1), (2, 0, 129)]])
def test_tiles_cover_their_rows(segs, group):
    t = ho.attn_tiles(segs, group)
    per = 32 if max(n for _, _, n in segs) * group <= 32 else 128
    want, row0 = set(), 0
    for b, p, n in segs:
        want |= {(i, row0, n, p, b) for i in range(-(-n * group // per))}
        row0 += n
    assert len(t) == len(want) and {tuple(r) for r in t.tolist()} == want
    last = [p + min(n, -(-(i + 1) * per // group)) for i, _, n, p, _ in t]
    assert (np.diff(last) <= 0).all()
