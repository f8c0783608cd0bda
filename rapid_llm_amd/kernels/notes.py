"""The launches of a piece of a step, noted while they are made, so that they can be made again for
layers that differ in nothing but their tensors (``ops.repeat_launches``).

Notes are a thread's own and live for the piece alone.  They keep every tensor that a noted launch was
given: the launches are made again with the same temporary tensors, which must not have gone to
somebody else meanwhile."""

from __future__ import annotations

import bisect
import contextlib
import ctypes
import threading

import numpy as np
import torch

# as csrc/repeat.hip lays them out
MAX_INTS, MAX_FLOATS = 32, 8
_CALL = np.dtype([("entry", "<i8"), ("ints", "<i8", (MAX_INTS,)), ("floats", "<f4", (MAX_FLOATS,))], align=True)


class _Thread(threading.local):
    notes: "Notes | None" = None


noting = _Thread()
#: The notes that threads are taking, none of them most of the time: a launch asks for its thread's own only where this is
#: not empty (a dozen questions a launch, 50 ns each for a thread's own, 10 for this).
taking: "list[Notes]" = []


class _Library:
    """A compiled library whose calls are noted."""

    def __init__(self, notes: "Notes", lib: ctypes.CDLL) -> None:
        self._notes, self._lib = notes, lib

    def __getattr__(self, name: str):
        entry = getattr(self._lib, name)

        def call(*args):
            self._notes.last = (name, entry, args)
            return entry(*args)

        return call


def _extent(t: torch.Tensor) -> int:
    """Bytes from a tensor's first element to behind its last."""
    return t.element_size() * (1 + sum((n - 1) * s for n, s in zip(t.shape, t.stride()))) if t.numel() else 0


class Notes:
    def __init__(self) -> None:
        self.calls: list[tuple] = []  # (the library's function, its arguments), as made
        self.tensors: list[torch.Tensor | None] = []
        self.last: tuple | None = None
        self.complete = True

    def library(self, lib: ctypes.CDLL) -> _Library:
        return _Library(self, lib)

    def made(self, what: str) -> None:
        """The call of the entry point ``what`` just made was a launch (calls that only ask a library something are not
        reported)."""
        if self.last is None or self.last[0] != what:
            self.complete = False  # of a library whose calls are not noted: the last noted call is another one
        else:
            self.calls.append(self.last[1:])
        self.last = None

    def give_up(self) -> None:
        """Something was launched that cannot be noted: nothing will be made again, and no tensor is kept for it."""
        self.complete = False
        self.last = None
        self.calls.clear()
        self.tensors.clear()

    def plan(self, tables, carried):
        """(calls, slots, table of pointers) for ``rl_repeat_calls``, or ``None`` where a call does not fit."""
        if not self.complete or not self.calls:
            return None
        pointers = [[t.data_ptr() for t in row] for row in tables]
        table = np.array(pointers, dtype=np.int64)
        if ((table ^ table[0]) & 15).any():
            return None  # which kernel runs may depend on where a tensor begins
        column: dict[int, tuple[int, int]] = {}
        spans = []
        for back, row in ((1, tables[0]), (0, tables[1])):
            for j, t in enumerate(row):
                at = pointers[1 - back][j]
                if at in column:
                    return None  # two layers share it: a pointer does not say whose it is
                column[at] = (j, back)
                spans.append((at, at + t.nbytes))
        spans.sort()
        starts = [s for s, _ in spans]
        before, after = (t.data_ptr() for t in carried)
        if carried[0].stride() != carried[1].stride() or carried[0].shape != carried[1].shape or (before ^ after) & 15:
            return None
        behind = before + _extent(carried[0])
        entries, all_ints, all_floats, slots = [], [], [], []
        for c, (entry, args) in enumerate(self.calls):
            ints, floats = [], []
            for arg in args:
                kind = type(arg)
                if kind is ctypes.c_void_p or arg is None:
                    value = 0 if arg is None else arg.value or 0
                    if value in column:
                        slots.append((c, len(ints), *column[value]))
                    elif before <= value < behind:
                        value += after - before  # (a launch may begin at any of its rows)
                    elif value:
                        i = bisect.bisect_right(starts, value) - 1
                        if i >= 0 and value < spans[i][1]:
                            return None
                    ints.append(value)
                elif kind is int or kind is bool:
                    ints.append(arg)
                elif kind is ctypes.c_float:
                    floats.append(arg.value)
                else:
                    return None
            if len(ints) > MAX_INTS or len(floats) > MAX_FLOATS:
                return None
            entries.append(ctypes.cast(entry, ctypes.c_void_p).value)
            all_ints.append(ints + [0] * (MAX_INTS - len(ints)))
            all_floats.append(floats + [0.0] * (MAX_FLOATS - len(floats)))
        calls = np.zeros(len(entries), dtype=_CALL)
        calls["entry"], calls["ints"], calls["floats"] = entries, all_ints, all_floats
        return calls, np.array(slots, dtype=np.int32).reshape(-1, 4), table


def unnoted() -> None:
    """To be called beside every kernel on a step's way that is not this package's (a product or a copy of torch's)."""
    if taking and noting.notes is not None:
        noting.notes.give_up()
        noting.notes = None


@contextlib.contextmanager
def taking_notes():
    """Note the launches that this thread makes inside the block."""
    outer, notes = noting.notes, Notes()
    taking.append(notes)
    noting.notes = notes
    try:
        yield notes
    finally:
        noting.notes = outer
        taking.remove(notes)
