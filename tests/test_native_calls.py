"""The native calls against the ctypes functions they stand for: the same
results and messages, and ctypes' own errors for arguments of other types."""

import ctypes

import pytest

from akv_amd import _lib


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
