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


def model(design="dense", **kw):
    import llm_np_cp_amd as L
    from llm_np_cp_amd.io.loader import LazyRandomWeights, random_weights
    from llm_np_cp_amd.models.registry import engine_class

    if design != "dense":
        cfg = L.preset_config(design)
        return engine_class(cfg)(cfg, LazyRandomWeights(cfg, seed=3),
                                 max_seq=256, max_batch=4, **kw)
    cfg = L.ModelConfig(
        model_type="llama", vocab_size=512, hidden_size=256,
        intermediate_size=768, num_hidden_layers=3, num_attention_heads=4,
        num_key_value_heads=2, head_dim=64)
    return engine_class(cfg)(cfg, random_weights(cfg, seed=3), max_seq=256,
                             max_batch=4, **kw)


def test_other_work_of_the_library_is_not_kept(ho):
    """A native call of many launches that has no place on the list."""
    c, m = Count(ho), model()

    def step():
        c.step()
        m._stack.forward(1, keys=1)

    assert ho.record(step) is None
    assert ho.record(lambda: (c.step(), m._stack.chunk_rows(9, 4))) is not None
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", ["bf16", "fp8"])
def test_steps_of_an_engine_are_kept(ho, dtype):
    """As launches: q, k and v, two a layer and the pick of one row, some a
    layer of a group; and they go on as a step by itself does."""
    m = model(dtype=dtype)
    m.prefill([1, 2, 3])
    ids = list(m.decode(9))
    assert type(m._graph).__name__ == "Tape" and len(m._graph) == 3 * 2 + 2
    m.prefill([1, 2, 3])
    assert list(m.decode(9, use_graph=False)) == ids
    m.prefill_batch([[1, 2, 3], [4, 5]])
    ids = m.decode_batch(9)
    assert type(m._graph).__name__ == "Tape" and len(m._graph) > 3 * 4
    m.prefill_batch([[1, 2, 3], [4, 5]])
    assert (m.decode_batch(9, use_graph=False) == ids).all()
    m.prefill_row(0, [1, 2, 3])
    m.prefill_row(1, [4, 5])
    m.decode_rows(2, 4)
    (g,) = m._bgraphs.values()
    assert type(g).__name__ == "Tape"


def test_steps_of_a_layer_list_are_kept(ho):
    m = model("garupel-2k")
    m.prefill([1, 2, 3])
    ids = list(m.decode(5))
    assert type(m._graph).__name__ == "Tape" and len(m._graph) > 40
    m.prefill([1, 2, 3])
    assert list(m.decode(5, use_graph=False)) == ids
    m.prefill_batch([[1, 2, 3], [4, 5]])
    m.decode_batch(5)
    assert type(m._graph).__name__ == "Tape" and len(m._graph) > 40


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
