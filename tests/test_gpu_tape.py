"""A step's launches, kept and made again: number and kinds of arguments,
blocks of arguments by value, what cannot be kept."""

import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


@pytest.fixture(scope="module")
def ho():
    from llm_np_cp_amd.ops import hip_ops
    return hip_ops


class Count:
    """h += W h (a launch of 26 numbers and 3 fractions) and n += 1."""

    def __init__(self, ho):
        self.ho = ho
        self.w = (torch.eye(64, device="cuda") * 2).bfloat16()
        self.h = torch.ones(64, dtype=BF, device="cuda")

    def step(self):
        self.ho.gemv(self.w, self.h, self.h, softcap=0.0)


@pytest.mark.parametrize("n", [1, 2, 11])
def test_replays(ho, n):
    c = Count(ho)
    tape = ho.record(c.step)
    assert len(tape) == 1
    tape.replay(n)
    tape.replay(1)
    torch.cuda.synchronize()
    assert (c.h == 2.0 ** (n + 2)).all()


def test_replays_on_the_current_stream(ho):
    c = Count(ho)
    tape = ho.record(c.step)
    s = torch.cuda.Stream()
    for _ in range(3):
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            torch.cuda._sleep(1000000)
            c.h.fill_(1.0)
            tape.replay(6)
        torch.cuda.current_stream().wait_stream(s)
        assert (c.h == 64.0).all()


def test_blocks_of_arguments_are_copied(ho):
    from llm_np_cp_amd.ops import hybrid_ops as hy
    x = torch.randn(8, 64, device="cuda")
    g = torch.ones(64, device="cuda")
    outs = [torch.zeros(8, 64, device="cuda") for _ in range(2)]

    def step():
        for o in outs:
            hy.norm_rows(x, g, o, 8, 64, 64, 1e-5)

    tape = ho.record(step)
    assert len(tape) == 2
    want = [o.clone() for o in outs]
    x.mul_(-1)
    tape.replay(5)
    for o, w in zip(outs, want):
        assert torch.equal(o, -w)


def test_what_is_no_launch_is_not_kept(ho):
    c = Count(ho)

    def more(what):
        def step():
            c.step()
            what()
        return step

    assert ho.record(more(lambda: c.h.mul_(1.0))) is None
    assert ho.record(more(lambda: torch.empty(3, device="cuda"))) is None
    s = torch.cuda.Stream()

    def elsewhere():
        with torch.cuda.stream(s):
            c.step()

    torch.cuda.synchronize()
    assert ho.record(more(elsewhere)) is None
    torch.cuda.synchronize()
    assert ho.record(lambda: None) is None
    # views are no work; the steps above did run
    assert ho.record(more(lambda: c.h[:3].view(3, 1))) is not None
    torch.cuda.synchronize()
    assert (c.h == 2.0 ** 5).all()


def test_only_this_thread_records(ho):
    import threading
    c, d = Count(ho), Count(ho)

    def step():
        c.step()
        t = threading.Thread(target=d.step)
        t.start()
        t.join()

    tape = ho.record(step)
    assert len(tape) == 1
    tape.replay(4)
    torch.cuda.synchronize()
    assert (c.h == 32.0).all() and (d.h == 2.0).all()


def test_a_launch_that_fails_is_named(ho):
    c = Count(ho)
    tape = ho.record(lambda: (c.step(), c.step()))
    tape._list[1].i[10] = 0               # K
    with pytest.raises(RuntimeError, match="launch 1 "):
        tape.replay(1)
