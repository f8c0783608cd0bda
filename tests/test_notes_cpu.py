"""Calls noted and made again from native code: arguments of every kind in any order, pointers out of the table."""

import ctypes

import pytest
import torch

from rapid_llm_amd.kernels import notes as notes_module
from rapid_llm_amd.kernels import ops

I, F, P = ctypes.c_int, ctypes.c_float, ctypes.c_void_p


def _entry(log, kinds):
    def body(*args):
        log.append(args)
        return 0

    return ctypes.CFUNCTYPE(I, *kinds)(body)


class _Lib:
    def __init__(self, **entries):
        self.__dict__.update(entries)


def _noted(lib, name, *args):
    with notes_module.taking_notes() as notes:
        getattr(notes.library(lib), name)(*args)
        ops._ok(0, name)
    return notes


def _again(notes, tables, carried):
    plan = notes.plan(tables, carried)
    assert plan is not None
    calls, slots, table = plan
    at = lambda a: P(a.ctypes.data)
    return ops.core().rl_repeat_calls(at(calls), len(calls), at(slots), len(slots), at(table), table.shape[1], 2, len(tables))


def test_calls_are_made_again_with_every_layers_tensors():
    # more integers than there are registers, floats between them, and as many of each as there may be
    kinds = [P, I, F, P, P, I, F, I, P, I, I, F, I, I, I, I, F, P, I, F, F, F, I, I, I, I, I, I, I, I, I, I, I, I, I, F, I, I, I, P]
    assert sum(k is not F for k in kinds) == notes_module.MAX_INTS and sum(k is F for k in kinds) == notes_module.MAX_FLOATS
    log = []
    lib = _Lib(rl_x=_entry(log, kinds))
    layers = [[torch.zeros(8), torch.zeros(3)] for _ in range(5)]
    x0, x1, other = torch.zeros(4), torch.zeros(4), torch.zeros(9)
    values = []
    for n, k in enumerate(kinds):
        values.append(F(n + 0.5) if k is F else P(other.data_ptr()) if k is P else -n if n % 2 else n)
    values[0], values[3], values[4], values[8] = (P(t.data_ptr()) for t in (layers[1][0], layers[0][1], x0, layers[1][1]))
    values[17] = None
    notes = _noted(lib, "rl_x", *values)
    assert _again(notes, layers, (x0, x1)) == 0
    assert len(log) == 4
    for place, args in enumerate(log[1:], start=2):
        want = list(log[0])
        want[0], want[3], want[4], want[8] = (t.data_ptr() for t in (layers[place][0], layers[place - 1][1], x1, layers[place][1]))
        assert list(args) == want


def test_pointers_into_the_carried_tensor_move_with_it():
    """A product cut into launches of fewer rows points at rows of what the layer before left, a view with rows apart too."""
    for wide, cols in ((torch.zeros(2, 6, 4), 4), (torch.zeros(2, 6, 10), 4)):
        x0, x1 = wide[0][:, :cols], wide[1][:, :cols]
        layers, log = [[torch.zeros(8)] for _ in range(4)], []
        behind = x0.data_ptr() + 4 * (5 * x0.stride(0) + cols)
        places = [x0.data_ptr(), x0[2:].data_ptr(), x0[5:].data_ptr() + 4]
        notes = _noted(_Lib(rl_x=_entry(log, [P, P, P, P])), "rl_x", *(P(p) for p in places), P(behind))
        assert _again(notes, layers, (x0, x1)) == 0
        step = x1.data_ptr() - x0.data_ptr()
        assert log[1:] == [(*(p + step for p in places), behind)] * 2
    x2 = torch.zeros(6, 8)[:, :4]  # rows elsewhere
    assert notes.plan(layers, (x0, x2)) is None


def test_a_call_that_fails_ends_it():
    log = []
    fail = ctypes.CFUNCTYPE(I, I)(lambda n: log.append(n) or (7 if len(log) > 2 else 0))
    notes = _noted(_Lib(rl_x=fail), "rl_x", 5)
    layers = [[torch.zeros(2)] for _ in range(9)]
    assert _again(notes, layers, (torch.zeros(1), torch.zeros(1))) == 7 and log == [5, 5, 5]


@pytest.mark.parametrize("why", ["inside", "shared", "argument", "many", "unknown", "asked", "address", "carried"])
def test_what_cannot_be_made_again(why):
    layers = [[torch.zeros(8)] for _ in range(4)]
    lib = _Lib(rl_x=lambda *a: 0)
    args = [P(layers[1][0].data_ptr())]
    if why == "inside":
        args = [P(layers[0][0].data_ptr() + 4)]  # the middle of a layer's tensor
    if why == "shared":
        layers[1][0] = layers[0][0]
    if why == "argument":
        args.append(1.5)  # neither a pointer nor an integer nor a float of the kernels' width
    if why == "many":
        args += [1] * notes_module.MAX_INTS
    notes = _noted(lib, "rl_x", *args)
    if why == "unknown":
        with notes_module.taking_notes() as notes:
            ops._ok(0, "a launch of a library that is not noted")
    if why == "asked":  # a question to a noted library, then a launch of one that is not
        with notes_module.taking_notes() as notes:
            notes.library(_Lib(rl_rows=lambda: 16)).rl_rows()
            ops._ok(0, "rl_x")
    carried = (torch.zeros(1), torch.zeros(1))
    if why == "address":  # a layer's tensor begins inside a unit of 16 bytes, the second's does not
        notes = _noted(_Lib(rl_x=_entry([], [P])), "rl_x", *args)
        assert notes.plan(layers, carried) is not None
        layers[3][0] = torch.zeros(9)[1:]
    if why == "carried":
        notes = _noted(_Lib(rl_x=_entry([], [P])), "rl_x", *args)
        carried = (torch.zeros(1), torch.zeros(2)[1:])
    assert notes.plan(layers, carried) is None


def test_every_launch_is_reported_under_its_entry_points_name():
    """What tells a launch from a question: a check's text is the name of the entry point whose code it checks."""
    import ast
    import inspect

    checks = [n for n in ast.walk(ast.parse(inspect.getsource(ops))) if isinstance(n, ast.Call) and getattr(n.func, "id", "") == "_ok"]
    named = [(n.args[0].func.attr, n.args[1].value) for n in checks]
    assert len(named) > 50 and all(entry == text for entry, text in named)


def test_notes_end_with_their_block_and_are_the_threads_own():
    import threading

    seen = []
    with notes_module.taking_notes():
        t = threading.Thread(target=lambda: seen.append(notes_module.noting.notes))
        t.start()
        t.join()
        assert notes_module.noting.notes is not None
    assert seen == [None] and notes_module.noting.notes is None


@pytest.mark.parametrize("what", ["library", "copy", "nothing"])
def test_what_is_not_this_packages_ends_the_notes(what):
    """A product or a copy of torch's between the launches: nothing is made again, and no tensor is kept for it."""
    layers = [[torch.zeros(8)] for _ in range(4)]
    lib, x = _Lib(rl_x=_entry([], [P])), torch.zeros(4, 8)
    with notes_module.taking_notes() as notes:
        notes.library(lib).rl_x(ops._p(layers[1][0]))
        ops._ok(0, "rl_x")
        if what == "library":
            ops.library_product(x, x)
        ops.whole_rows(x[:, :4] if what == "copy" else x)
        notes.library(lib).rl_x(ops._p(x))
        ops._ok(0, "rl_x")
    left = what == "nothing"
    assert (notes.plan(layers, (torch.zeros(1), torch.zeros(1))) is not None) == left
    assert notes.complete == left and bool(notes.tensors) == left


def test_launches_outside_of_notes_do_not_look_for_a_threads_own(monkeypatch):
    class Nobody:
        @property
        def notes(self):
            raise AssertionError("looked for")

    with notes_module.taking_notes():
        pass
    monkeypatch.setattr(ops, "noting", Nobody())
    assert not notes_module.taking
    ops.core(), ops._p(torch.zeros(1)), ops._ok(0, "rl_x"), ops.library_product(torch.zeros(2, 2), torch.zeros(2, 2))


def test_a_host_whose_calls_are_not_known_repeats_nothing(monkeypatch):
    """The library then says that a call holds nothing: the layers make their own launches."""
    layers = [[torch.zeros(8)] for _ in range(4)]
    log = []
    notes = _noted(_Lib(rl_x=_entry(log, [P])), "rl_x", P(layers[1][0].data_ptr()))
    carried = (torch.zeros(1), torch.zeros(1))
    assert ops.repeat_launches(notes, layers, carried) and len(log) == 3
    nowhere = _Lib(rl_repeat_max_ints=lambda: 0, rl_repeat_max_floats=lambda: 0, rl_repeat_calls=lambda *args: 1)
    monkeypatch.setattr(ops, "core", lambda: nowhere)
    assert not ops.repeat_launches(notes, layers, carried) and len(log) == 3
