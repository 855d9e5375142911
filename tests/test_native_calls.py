"""The native calls against the ctypes functions they stand for: the same
results and messages, and ctypes' own errors for arguments of other types; the
module is this interpreter's, and ctypes stands in where there is none."""

import ctypes
import sys
import sysconfig

import pytest

import akv_amd
from akv_amd import _lib, build


def _zeros(fn):
    return [None if t is _lib.c_void_p else 0.0 if t is ctypes.c_float else 0 for t in fn.argtypes]


@pytest.mark.parametrize("value", [0, -1, 3])
def test_same_results_as_ctypes(value):
    calls, lib = _lib.calls(), _lib.load()
    for name in calls.names():
        fn = getattr(lib, name)
        args = [value if t in (ctypes.c_int32, ctypes.c_int64) else a for t, a in zip(fn.argtypes, _zeros(fn))]
        # no call here passes its checks with null pointers and work to do
        want = fn(*args)
        message = _lib.last_error()
        assert getattr(calls, name)(*args) == want, name
        assert _lib.last_error() == message


def test_other_types_meet_ctypes():
    calls, lib = _lib.calls(), _lib.load()
    args = _zeros(lib.akv_build_indptr)
    for bad in ([1.5] + args[1:], args[:1] + [1.5] + args[2:]):
        with pytest.raises(ctypes.ArgumentError):
            calls.akv_build_indptr(*bad)
    with pytest.raises(TypeError):
        calls.akv_build_indptr(*args[:-1])
    # booleans and integers past 64 bits' sign are integers, as for ctypes
    assert calls.akv_decode_attention_workspace_bytes(True, 1, 64, 1) == lib.akv_decode_attention_workspace_bytes(1, 1, 64, 1)
    assert calls.akv_decode_attention_workspace_bytes(2 ** 32 + 1, 1, 64, 1) == \
        lib.akv_decode_attention_workspace_bytes(2 ** 32 + 1, 1, 64, 1)


def test_module_is_named_for_the_interpreter():
    assert build.NATIVE.name == "_native" + sysconfig.get_config_var("EXT_SUFFIX")
    assert _lib.calls().__file__ == str(build.NATIVE)


def test_ctypes_without_the_module(monkeypatch):
    monkeypatch.setattr(_lib, "_calls", None)
    monkeypatch.delattr(akv_amd, "_native", raising=False)
    monkeypatch.setitem(sys.modules, "akv_amd._native", None)  # as if it could not be imported
    with pytest.warns(RuntimeWarning, match="native calls are not built"):
        calls = _lib.calls()
    assert calls is _lib.load() and _lib.calls() is calls
    assert calls.akv_decode_attention_workspace_bytes(1, 1, 64, 1) > 0


def test_build_without_python_headers(monkeypatch, tmp_path, capsys):
    """The library is built and the module left out."""
    ran = []
    monkeypatch.setattr(build, "_run", lambda cmd: ran.append(cmd) or "")
    monkeypatch.setattr(build.os, "replace", lambda a, b: None)
    monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    assert build.build() == build.LIBRARY
    assert "no Python.h" in capsys.readouterr().out
    assert not any("native.cpp" in str(a) for cmd in ran for a in cmd)
    assert any(str(a).endswith("libakv_amd.so.tmp") for cmd in ran for a in cmd)
