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
    for l, signatures in ((_lib.lib(), _lib.SIGNATURES), (_lib.mixers_lib(), _lib.MIXERS_SIGNATURES)):
        bound = [n for n in signatures if type(getattr(l, n)).__name__ == "builtin_function_or_method"]
        assert 2 * len(bound) > len(signatures)
        assert all(getattr(l, n).__name__ == n for n in bound)


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
