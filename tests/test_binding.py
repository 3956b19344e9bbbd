"""The native call path: what it converts itself and what it leaves to ctypes give the same calls."""
import ctypes
import importlib
import threading

import numpy as np
import pytest

from minit_amd import lib
from minit_amd.core.object import Object

table = importlib.import_module("minit_amd.core.dispatch")   # the package re-exports the function of that name

SIZES = (1, 4096, 4096, 128, 4)


def test_the_module_is_the_path():
    assert lib.call is lib._binding.call


@pytest.mark.parametrize("sizes", [SIZES, (16, 5120, 13696, 128, 8), (64, 4096, 14336, 32, 4), (1, 4096, 4100, 128, 4),
                                   (-1, 4096, 4096, 128, 4), (2 ** 32 + 1, 4096, 4096, 128, 4), (2 ** 70 + 1, 4096, 4096, 128, 4)])
def test_numbers_as_ctypes_takes_them(sizes):
    """Widths, signs and the reduction of numbers that do not fit."""
    lib.cdll()
    expected = lib._call_general("mh_gptq_workspace_bytes", *sizes)
    assert lib.call("mh_gptq_workspace_bytes", *sizes) == expected
    assert lib.call("mh_gptq_workspace_bytes", *(ctypes.c_int(s) for s in sizes)) == expected
    if max(sizes) < 2 ** 31:
        assert lib.call("mh_gptq_workspace_bytes", *(np.int64(s) for s in sizes)) == expected


def test_what_is_refused():
    lib.cdll()
    for call in (lib.call, lib._call_general):
        with pytest.raises(TypeError):
            call("mh_gptq_workspace_bytes", *SIZES[:-1])
        with pytest.raises(ctypes.ArgumentError):
            call("mh_gptq_workspace_bytes", 1.0, *SIZES[1:])
        with pytest.raises(ctypes.ArgumentError):
            call("mh_softmax_causal", 2.5, 256, 256, 1, 2, 7, 3, 1.0, 0)
        with pytest.raises(lib.HipError, match=r"mh_softmax_causal failed \(1\): .*t=7 must equal"):
            call("mh_softmax_causal", None, 256, 256, 1, 2, 7, 3, 1, 0)
        with pytest.raises(AttributeError):
            call("mh_no_such_function")
    with pytest.raises(TypeError):
        lib.call(*[], **{"name": "mh_abi_version"})


def test_status_messages_are_the_callers_own():
    """The message of a failed call belongs to the thread that made it."""
    seen = []

    def other():
        with pytest.raises(lib.HipError, match="bits must be 4 or 8") as e:
            lib.call("mh_gptq_unpack", None, 256, 256, 4, 4, 0, 5)
        seen.append(str(e.value))
    threads = [threading.Thread(target=other) for _ in range(4)]
    with pytest.raises(lib.HipError, match="t=7 must equal"):
        lib.call("mh_softmax_causal", None, 256, 256, 1, 2, 7, 3, 1.0, 0)
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(seen) == 4


def test_a_failure_elsewhere_leaves_the_message():
    """Between the status of a call and the question for its message, another thread fails with another message."""
    failed, other_failed = threading.Event(), threading.Event()
    seen = []

    def first():
        assert lib.cdll().mh_softmax_causal(None, 256, 256, 1, 2, 7, 3, 1.0, 0) != 0
        failed.set()
        assert other_failed.wait(30)
        seen.append(lib.last_error())

    def second():
        assert failed.wait(30)
        with pytest.raises(lib.HipError, match="bits must be 4 or 8"):
            lib.call("mh_gptq_unpack", None, 256, 256, 4, 4, 0, 5)
        other_failed.set()
    threads = [threading.Thread(target=f) for f in (first, second)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(seen) == 1 and "t=7 must equal" in seen[0]


def test_signatures_of_another_build(monkeypatch):
    """Where the prototypes are not the ones the module was compiled for, calls take the path that converts by the prototypes."""
    entries = lib._entries(lib.cdll())
    assert lib._binding.bind(entries) == 0
    name = "mh_gptq_workspace_bytes"
    reached = []
    monkeypatch.setitem(lib._functions, name, lambda *args: reached.append(args))
    lib.call(name, *SIZES)
    assert not reached
    try:
        for signature in ("Liiii", "Liiiiii", "Liiiif", "iiiiii"):
            assert lib._binding.bind({**entries, name: (entries[name][0], signature)}) == 1
            lib.call(name, *SIZES)
            assert reached.pop() == SIZES and not reached
        with pytest.raises(Exception):
            lib._binding.bind({**entries, name: entries[name][0]})
    finally:
        lib._binding.bind(entries)


class _Op(Object):
    def type(self):
        return _Op


class _Value(Object):
    def type(self):
        return _Value


@pytest.mark.parametrize("dispatch", [table.dispatch, table._dispatch])
def test_dispatch_native_and_python(dispatch, monkeypatch):
    monkeypatch.setattr(table, "DISPATCH_TABLE", list(table.DISPATCH_TABLE))
    held = dict(table.DISPATCH_CACHE)
    try:
        with pytest.raises(AssertionError, match="no matching function"):
            dispatch(_Op(), _Value())
        calls = []

        @table.register_dispatch()
        def rule(op: _Op, x: _Value):
            calls.append(x)
            return (x,)
        value = _Value()
        assert dispatch(_Op(), value) == (value,) and dispatch(_Op(), value) == (value,) and calls == [value, value]

        @table.register_dispatch(priority=2)   # clears the cache: the better rule is found
        def other(op: _Op, x: _Value):
            raise ValueError("from the rule")
        with pytest.raises(ValueError, match="from the rule"):
            dispatch(_Op(), value)
        with pytest.raises(AttributeError):
            dispatch(_Op(), 3)
    finally:
        table.DISPATCH_CACHE.clear()
        table.DISPATCH_CACHE.update(held)
