"""The step calls of the Python binding (binding.cpp) against ctypes: every one of them is bound to a function that
records its arguments, with the argument types that hip.SIGNATURES declares, and has to hand over what ctypes
hands over."""
import ctypes as C
import importlib.util
import threading
import types as _types

import numpy as np
import pytest

from cwick_amd import build, hip


class Tensor:
    """What a device tensor is to the binding."""

    def __init__(self, address, cuda=True, dense=True):
        self.address, self.is_cuda, self.dense = address, cuda, dense

    def is_contiguous(self):
        return self.dense

    def data_ptr(self):
        return self.address


class Stream:
    """What torch.cuda.Stream is to ctypes."""

    def __init__(self, address):
        self._as_parameter_ = C.c_void_p(address)


def _recorder(name):
    res, types = hip.SIGNATURES["cwick_hip_" + name]
    seen = []

    def record(*args):
        seen.append(args)
        return len(seen)

    fn = C.CFUNCTYPE(res, *types)(record)
    return fn, types, seen


def _module():
    """The extension by itself: it does not need libcwick_hip.so (which is loaded after torch or not at all)."""
    spec = importlib.util.spec_from_file_location("_cwick_calls", hip.CALLS_PATH)
    m = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(m)
    return m


NAMES = _module().names()


@pytest.mark.parametrize("name", NAMES)
def test_arguments_arrive_as_through_ctypes(name):
    fn, types, seen = _recorder(name)
    call = _module().bind(name, C.cast(fn, C.c_void_p).value)
    ints = (7, -3, 2 ** 31 + 5, 2 ** 63 - 1, -2 ** 63, True, np.int64(12), 2 ** 64 + 9)
    arrays = [np.arange(4 + i, dtype=np.float32) for i in range(len(types))]
    for turn in range(len(ints)):
        given, plain = [], []
        for i, t in enumerate(types):
            if t is C.c_void_p:
                kind = (turn + i) % 3
                a = None if kind == 0 else 0x7F0000001000 + 64 * i if kind == 1 else arrays[i].ctypes.data
                plain.append(a)
                device = Stream if i == len(types) - 1 else Tensor
                given.append(a if kind < 2 else device(a) if name.endswith("_dev") else arrays[i])
            elif t is C.c_float:
                plain.append((0.125, 3, -1.0, 1e300, np.float32(0.1), float("nan"), True, 0.1)[turn])
                given.append(plain[-1])
            else:
                plain.append(ints[(turn + i) % len(ints)])
                given.append(plain[-1])
        assert call(*given) == 2 * turn + 1
        assert fn(*plain) == 2 * turn + 2
        assert repr(seen[-2]) == repr(seen[-1])


def test_what_is_no_argument_is_refused():
    fn, types, seen = _recorder("topk_dev")
    call = _module().bind("topk_dev", C.cast(fn, C.c_void_p).value)
    ok = [Tensor(64), 1, 2, 3, Tensor(128), None]
    assert call(*ok) == 1 and seen[-1] == (64, 1, 2, 3, 128, None)
    assert call(*ok[:5], C.c_void_p(256)) == 2 and seen[-1][-1] == 256       # a stream as ctypes has it
    for at, bad, error in ((0, Tensor(64, cuda=False), AssertionError), (4, Tensor(64, dense=False), AssertionError),
                           (0, np.zeros(3), AttributeError), (1, 2.5, TypeError), (1, None, TypeError), (2, "3", TypeError)):
        with pytest.raises(error):
            call(*(ok[:at] + [bad] + ok[at + 1:]))
    with pytest.raises(TypeError):
        call(*ok[:5])
    with pytest.raises(TypeError):
        _module().bind("kv_write_f32", C.cast(fn, C.c_void_p).value)(None, 0, 1, object(), None)
    with pytest.raises(ValueError):
        _module().bind("kv_write_f32", C.cast(fn, C.c_void_p).value)(None, 0, 1, np.zeros((4, 4))[:, ::2], None)
    with pytest.raises(ValueError):
        _module().bind("no_such_call", 1)
    assert len(seen) == 2


def test_a_stream_is_what_ctypes_takes_as_one():
    """The last argument of a call on device memory: all that ctypes makes a void pointer of, and nothing else.  A tensor
    there would be a stream whose state is the tensor's bytes."""
    fn, types, seen = _recorder("topk_dev")
    call = _module().bind("topk_dev", C.cast(fn, C.c_void_p).value)
    head = [64, 1, 2, 3, 128]
    block = C.create_string_buffer(8)
    for stream in (None, 0, 4096, C.c_void_p(), C.c_void_p(4096), Stream(0), Stream(4096), C.cast(block, C.POINTER(C.c_char)), block):
        assert call(*head, stream) == fn(*head, stream) - 1
        assert seen[-1] == seen[-2]
    n = len(seen)
    for bad in (Tensor(64), object(), 2.5, np.zeros(3), np.int64(4096)):
        for f in (call, fn):
            with pytest.raises(C.ArgumentError):
                f(*head, bad)
    with pytest.raises(AttributeError):                     # and a pointer is no tensor
        call(C.c_void_p(64), *head[1:], None)
    assert len(seen) == n


@pytest.mark.parametrize("at,bad", [(1, 2.5), (1, None), (2, "3"), (3, np.zeros(2))])
def test_refused_arguments_raise_what_ctypes_raises(at, bad):
    fn, types, seen = _recorder("topk_dev")
    call = _module().bind("topk_dev", C.cast(fn, C.c_void_p).value)
    given = [64, 1, 2, 3, 128, None]
    given[at] = bad
    for f in (call, fn):
        with pytest.raises(C.ArgumentError):
            f(*given)
    fn, types, seen = _recorder("gqa_decode")
    call = _module().bind("gqa_decode", C.cast(fn, C.c_void_p).value)
    for bad in ("0.5", None, 10 ** 400):
        for f in (call, fn):
            with pytest.raises(C.ArgumentError):
                f(64, 1, None, 2, bad, None)
    assert not seen


def test_the_interpreter_runs_during_a_call():
    """A call that waits (here: for another Python thread) does not hold the interpreter's lock."""
    go = threading.Event()
    res, types = hip.SIGNATURES["cwick_hip_topk_dev"]
    fn = C.CFUNCTYPE(res, *types)(lambda *a: int(go.wait(30)))
    call = _module().bind("topk_dev", C.cast(fn, C.c_void_p).value)
    t = threading.Timer(0.05, go.set)
    t.start()
    assert call(None, 1, 2, 3, None, None) == 1
    t.join()


@pytest.mark.parametrize("name", NAMES)
def test_calls_go_through_ctypes_without_the_extension(name, monkeypatch, tmp_path):
    """The extension is built for one interpreter; the library serves any other through ctypes."""
    fn, types, seen = _recorder(name)
    bound = _module().bind(name, C.cast(fn, C.c_void_p).value)
    monkeypatch.setattr(hip, "CALLS_PATH", str(tmp_path / "missing.so"))
    monkeypatch.setattr(hip, "_c", None)
    monkeypatch.setattr(hip, "_lib", _types.SimpleNamespace(**{"cwick_hip_" + name: fn}))
    call = getattr(hip._calls(), name)
    arrays = [np.arange(4 + i, dtype=np.float32) for i in range(len(types))]
    for turn in range(3):
        given = []
        for i, t in enumerate(types):
            if t is C.c_void_p:
                device = Stream if i == len(types) - 1 else Tensor
                given.append((None, 4096 + i, device(64 * i + 64) if name.endswith("_dev") else arrays[i])[(turn + i) % 3])
            else:
                given.append(0.25 if t is C.c_float else 11 + i)
        assert call(*given) == bound(*given) - 1
        assert repr(seen[-2]) == repr(seen[-1])


def test_the_library_builds_without_the_headers_of_python(monkeypatch, tmp_path, capsys):
    monkeypatch.setattr(build, "CALLS", str(tmp_path / "calls.so"))
    with monkeypatch.context() as m:
        m.setattr(build.sysconfig, "get_path", lambda name: str(tmp_path))
        build._build_calls(force=True)
    with monkeypatch.context() as m:
        m.setenv("CXX", str(tmp_path / "no-compiler"))
        build._build_calls(force=True)
    out = capsys.readouterr().out
    assert "no Python.h: the step calls" in out and "no-compiler: the step calls" in out
    assert not (tmp_path / "calls.so").exists()
