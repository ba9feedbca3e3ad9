"""What of a step can be kept: by name and by kind of argument."""

import ctypes

import pytest

from llm_np_cp_amd.ops import hip_ops, hybrid_ops, tape

NATIVE = sorted(set(hip_ops._SIGS) |
                {n for s in hybrid_ops._SIGS.values() for n in s})


def add(argtypes, args):
    fn = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: 0)
    fn.argtypes = argtypes
    fn.__name__ = "launch_native"
    t = tape.Tape(None)
    t.add(fn, args)
    return t


@pytest.mark.parametrize("name", NATIVE)
def test_by_name(name):
    """A launch is noted, a question is not work, and whatever else the
    libraries have makes the step one that is not kept."""
    rec = tape._Recorder(tape.Tape(None), 0)

    def fn():
        pass

    got = tape.noted(name, fn, rec)
    if name.startswith("launch_"):
        assert got is not fn and rec.other is None
    else:
        assert got is fn
        assert rec.other == (None if name in tape.ASKS else name)
    assert tape.noted(name, fn) is fn         # where nothing is recorded


def test_arguments():
    class Block(ctypes.Structure):
        _fields_ = [("a", ctypes.c_int), ("b", ctypes.c_float)]

    v, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    b = Block(3, 0.5)
    t = add([v, i, f, v, v, v, i, v],
            [1 << 63, -2, 0.25, None, ctypes.byref(b), b,
             ctypes.c_int(7), 9])
    c = t._list[0]
    assert c.n == 7 and list(c.f)[0] == 0.25
    assert [c.i[0], c.i[1], c.i[2], c.i[5], c.i[6]] == \
        [-(1 << 63), -2, 0, 7, 9]
    b.a = 4                                   # by value
    for at in (c.i[3], c.i[4]):
        assert Block.from_address(at).a == 3


@pytest.mark.parametrize("argtypes,args", [
    ([ctypes.c_double, ctypes.c_void_p], [0.5, 1]),
    ([ctypes.c_void_p, ctypes.c_void_p], [ctypes.c_double(0.5), 1]),
    ([ctypes.c_void_p, ctypes.c_void_p], [0.5, 1]),
    ([ctypes.c_void_p, ctypes.c_void_p], ["text", 1]),
    ([ctypes.c_void_p, ctypes.c_void_p],
     [ctypes.pointer(ctypes.c_int(3)), 1]),
    ([ctypes.c_void_p, ctypes.c_void_p], [ctypes.byref(ctypes.c_int(3)), 1]),
    ([ctypes.c_void_p], [1, 2]),
    ([ctypes.c_int] * 40, [1] * 40),
    ([ctypes.c_float] * 9, [1.0] * 9)])
def test_arguments_that_cannot_be_kept(argtypes, args):
    with pytest.raises(ValueError):
        add(argtypes, args)
