"""Calls of the C entry points through typed Python functions (csrc_torch/entry_calls.cpp) against the same calls through ctypes: the same results for
plain numbers, and the same exceptions and results for whatever else a caller may pass.  Only entry points that answer on the host are called."""
import ctypes

import pytest

from aphrodite_engine_amd import _lib


def plain(name):
    signatures, path = (_lib.SIGNATURES, _lib.LIB_PATH) if name in _lib.SIGNATURES else (_lib.MIXERS_SIGNATURES, _lib.MIXERS_LIB_PATH)
    fn = getattr(ctypes.CDLL(path), name)
    fn.restype, fn.argtypes = signatures[name]
    return fn


def typed(name):
    return getattr(_lib.lib() if name in _lib.SIGNATURES else _lib.mixers_lib(), name)


def outcome(fn, args):
    try:
        return fn(*args)
    except Exception as e:
        return type(e), str(e)


def test_the_entry_points_are_bound():
    calls = _lib._entry_calls()
    assert len(calls.names()) == len(set(calls.names())) >= 170
    for name in calls.names():
        fn = typed(name)
        assert type(fn).__name__ == "builtin_function_or_method" and fn.__name__ == name


@pytest.mark.parametrize("name", ["aphro_dense_rows_slab_floats", "aphro_rms_norm", "aphro_distance_bias_attention"])
def test_other_types_than_the_module_was_built_with(name):
    """Signatures and module that do not agree in one type, or in their number: the name stays with ctypes."""
    calls, fn = _lib._entry_calls(), plain(name)
    at, types = ctypes.cast(fn, ctypes.c_void_p).value, _lib._letters(fn.restype, fn.argtypes)
    assert calls.bind(name, at, fn, types).__name__ == name
    for i in range(len(types)):
        for other in "PilLf?":
            if other != types[i]:
                assert calls.bind(name, at, fn, types[:i] + other + types[i + 1:]) is None
    assert calls.bind(name, at, fn, types + "P") is None and calls.bind(name, at, fn, types[:-1]) is None


def test_a_moved_signature_keeps_ctypes():
    name = "aphro_dense_rows_slab_floats"
    l = ctypes.CDLL(_lib.LIB_PATH)
    moved = (ctypes.c_int, [ctypes.c_float] + _lib.SIGNATURES[name][1][1:])
    getattr(l, name).restype, getattr(l, name).argtypes = moved
    _lib._bind_calls(l, {name: moved})
    assert not type(getattr(l, name)).__name__.startswith("builtin")


def test_built_for_another_python(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "ENTRY_CALLS_PATH", str(tmp_path / "aphrodite_entry_calls.so"))
    l = ctypes.CDLL(_lib.LIB_PATH)
    _lib._bind_calls(l, {"aphro_rms_norm": _lib.SIGNATURES["aphro_rms_norm"]})
    assert not type(l.aphro_rms_norm).__name__.startswith("builtin")


SLAB = (32, 4096, 4096, 4096, 4096, -1)


@pytest.mark.parametrize("args", [
    SLAB, (1, 128, 4096, 128, 4096, -1), (True, 4096, 4096, 4096, 4096, -1), (32 + 2**64, ) + SLAB[1:], SLAB[:-1], (), SLAB + (0, ),
    (32.0, ) + SLAB[1:], ("32", ) + SLAB[1:], (None, ) + SLAB[1:], (ctypes.c_int64(32), ) + SLAB[1:],
])
def test_whole_numbers_and_everything_else(args):
    name = "aphro_dense_rows_slab_floats"
    assert outcome(typed(name), args) == outcome(plain(name), args)


@pytest.mark.parametrize("pointer", [None, 0, 256, ctypes.c_void_p(256), ctypes.c_void_p(), "256", 2.0, -1])
@pytest.mark.parametrize("rows,k", [(0, 1024), (4, 1000)])
def test_pointers(pointer, rows, k):
    name = "aphro_silu_and_mul_pack_slabs"        # refuses 1000 columns and returns at once without rows
    args = (pointer, 2, 256, None, rows, k, _lib.F16, None)
    assert outcome(typed(name), args) == outcome(plain(name), args)


def test_floats():
    name = "aphro_rms_norm"
    types = _lib.SIGNATURES[name][1]
    at = [i for i, t in enumerate(types) if t is ctypes.c_float]
    assert at
    for value in (1e-6, 1, True, 10**400, None, "1", ctypes.c_float(1.0)):
        args = [0] * len(types)                   # no rows: returns, or refuses, on the host
        args[at[0]] = value
        assert outcome(typed(name), args) == outcome(plain(name), args)
