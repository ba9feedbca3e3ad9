"""What the native launcher of a prompt's rows refuses before it launches
anything: rows beyond its scratch, positions and pools beyond the cache."""

import numpy as np
import pytest
import torch

from llm_np_cp_amd.ops import hip_ops as ho

ROWS, S, POOLS = 40, 24, 3


@pytest.fixture(scope="module", autouse=True)
def _build():
    from csrc.build import ensure_built
    ensure_built(names=["llmops"])


@pytest.fixture
def stack(monkeypatch):
    monkeypatch.setattr(ho, "_stream", lambda: 0)
    return ho.Stack([{}], rows=ROWS, S=S, pools=POOLS, mfma=1, H=64, nh=1,
                    kvh=1, hd=64)


def refused(call):
    with pytest.raises(RuntimeError, match="hipError_t=1$"):
        call()


def packed(M, most, n=1):
    return dict(rows=torch.zeros(2 * M, dtype=torch.int32),
                tiles=torch.zeros(n, 5, dtype=torch.int32), most=most)


@pytest.mark.parametrize("M,keys,kw", [
    (0, 1, {}), (ROWS + 1, S, packed(ROWS + 1, 4)), (S + 1, S, {}),
    (2, S + 1, {}), (2, S + 1, packed(2, 1)), (2, 2, dict(pool=-1)),
    (2, 2, dict(pool=POOLS)), (2, 2, packed(2, 0)), (2, 2, packed(2, 3)),
    (2, 2, dict(first=-1)), (2, 2, dict(last=2))])
def test_layers_refuse(stack, M, keys, kw):
    refused(lambda: stack.forward(M, keys, **kw))


@pytest.mark.parametrize("M,pos0", [(0, 0), (ROWS + 1, 0), (1, -1), (1, S)])
def test_embedding_refuses(stack, M, pos0):
    refused(lambda: stack.embed(np.zeros(M, np.int32), M, pos0))
    refused(lambda: stack.embed(torch.zeros(M, dtype=torch.int32), M, pos0))


def test_lists_are_as_long_as_the_chunk(stack):
    with pytest.raises(AssertionError):
        stack.embed(torch.zeros(1, dtype=torch.int32), 2, 0)
    with pytest.raises(AssertionError):
        stack.forward(3, 3, **packed(2, 2))


# the layers of no list: what the limits let through reaches the end
@pytest.mark.parametrize("M,keys,kw", [
    (S, S, dict(pool=POOLS - 1)), (1, S, {}), (ROWS, S, packed(ROWS, S))])
def test_layers_take_what_fits(stack, M, keys, kw):
    stack.forward(M, keys, first=1, last=1, **kw)
