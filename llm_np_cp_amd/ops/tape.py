"""A decode step's launches, kept as they were made, and made again from
native code (csrc/tape.hip) as often as asked.

``record(step)`` runs ``step`` for real and keeps every launch that it makes
through the kernel libraries: the launcher and its arguments, blocks of
arguments by value.  What it cannot keep makes it return None, and the caller
captures the step instead: an operation of torch that is no view (new memory
among them), a launch on another stream, any other native function but those
that only answer, an argument that is neither whole number, pointer, block nor
c_float.  The addresses are those of the
engine's own buffers, as in a captured graph.
"""

from __future__ import annotations

import ctypes
import threading

import torch
from torch.utils._python_dispatch import TorchDispatchMode

INTS, FLOATS = 32, 8
# native functions that enqueue nothing
ASKS = frozenset(("row_gemm_plan", "chain_slots", "stack_chunk_rows",
                  "attn_prefill_plan", "gemm_prompt_plan", "expert_gemm_plan"))
_local = threading.local()


class _Call(ctypes.Structure):
    _fields_ = [("fn", ctypes.c_void_p), ("n", ctypes.c_long),
                ("i", ctypes.c_long * INTS), ("f", ctypes.c_float * FLOATS)]


def _word(v, held) -> int:
    """An argument as eight bytes; blocks of arguments are copied."""
    if v is None:
        return 0
    if isinstance(v, int):
        return v
    obj = getattr(v, "_obj", v)          # ctypes.byref
    if isinstance(obj, (ctypes.Structure, ctypes.Array)):
        copy = type(obj).from_buffer_copy(obj)
        held.append(copy)
        return ctypes.addressof(copy)
    if obj is v and isinstance(getattr(v, "value", v), (int, type(None))):
        return v.value or 0
    raise ValueError(f"an argument that is {v!r}")


class Tape:
    """Launches in their order.  ``replay(n)`` makes all of them n times on
    the current stream."""

    def __init__(self, lib):
        self._lib, self._list, self._held = lib, [], []
        self._calls = None

    def __len__(self):
        return len(self._list)

    def add(self, fn, args) -> None:
        c, ints, floats = _Call(), [], []
        for t, v in zip(fn.argtypes, args):
            if t is ctypes.c_float:
                floats.append(float(getattr(v, "value", v)))
            elif t in (ctypes.c_double, ctypes.c_longdouble):
                raise ValueError(f"{fn.__name__}: a fraction of more bits")
            else:
                ints.append(_word(v, self._held))
        if len(args) != len(fn.argtypes) or len(ints) > INTS or \
                len(floats) > FLOATS:
            raise ValueError(f"{fn.__name__}: {len(args)} arguments")
        c.fn = ctypes.cast(fn, ctypes.c_void_p).value
        c.n = len(ints)
        for k, v in enumerate(ints):
            # as an unsigned address or a signed number
            c.i[k] = v - (1 << 64) if v >= 1 << 63 else v
        c.f[:len(floats)] = floats
        self._list.append(c)

    def replay(self, times: int = 1) -> None:
        n, at = len(self._list), ctypes.c_int(-1)
        if self._calls is None:
            self._calls = (_Call * n)(*self._list)
        err = self._lib.tape_run(self._calls, n, times,
                                 torch.cuda.current_stream().cuda_stream,
                                 ctypes.byref(at))
        if err != 0:
            raise RuntimeError(f"launch {at.value} of a recorded step "
                               f"failed: hipError_t={err}")


class _Recorder(TorchDispatchMode):
    """Notes what torch itself does besides."""

    def __init__(self, tape, stream):
        super().__init__()
        self.tape, self.stream, self.other = tape, stream, None

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        if not func.is_view:
            self.other = self.other or str(func)
        return func(*args, **(kwargs or {}))

    def launch(self, fn):
        def call(*args):
            if args[-1] != self.stream:
                self.other = self.other or "another stream"
            try:
                self.tape.add(fn, args)
            except ValueError as e:
                self.other = self.other or str(e)
            return fn(*args)
        return call


class _Library:
    """A kernel library whose launches are noted."""

    def __init__(self, lib, recorder):
        self._lib, self._recorder = lib, recorder

    def __getattr__(self, name):
        return noted(name, getattr(self._lib, name), self._recorder)


def noted(name: str, fn, recorder=None):
    """fn, or while this thread records a step and fn launches, fn noted.
    Work under another name cannot be kept, and then the step is not."""
    recorder = recorder or getattr(_local, "recorder", None)
    if recorder is None or name in ASKS:
        return fn
    if name.startswith("launch_"):
        return recorder.launch(fn)
    recorder.other = recorder.other or name
    return fn


def library(lib):
    recorder = getattr(_local, "recorder", None)
    return lib if recorder is None else _Library(lib, recorder)


def record(step, lib):
    """Runs step() and returns the Tape of it, or None (the step did run)
    where it was more than launches.  lib: the library with tape_run."""
    tape = Tape(lib)
    rec = _Recorder(tape, torch.cuda.current_stream().cuda_stream)
    _local.recorder = rec
    try:
        with rec:
            step()
    finally:
        _local.recorder = None
    return tape if rec.other is None and len(tape) else None
