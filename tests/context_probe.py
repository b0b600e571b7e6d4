"""Read-only view of a solver's plan (tests/cpp/context_probe.cpp)."""
import ctypes as C
import os

import numpy as np

_lib = None


def _probe():
    global _lib
    if _lib is None:
        _lib = C.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "bin", "libcontext_probe.so"))
        _lib.probe_ways.argtypes = _lib.probe_graphs.argtypes = [C.c_void_p]
        _lib.probe_items.argtypes = [C.c_void_p, C.c_void_p, C.c_int]
    return _lib


def ways(solver) -> int:
    return _probe().probe_ways(solver._h)


def graphs(solver) -> int:
    return _probe().probe_graphs(solver._h)


def item_rows(solver) -> np.ndarray:
    """Rows of each item of a step's main launch (negative: columns of a transposed one)."""
    n = _probe().probe_items(solver._h, None, 0)
    out = np.zeros(max(n, 1), np.int32)
    _probe().probe_items(solver._h, out.ctypes.data, n)
    return out[:n]
