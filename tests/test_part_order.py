"""The vertex numbering of the resident PCG (sk_part_order, host only): a permutation in contiguous, non-empty parts
of at most a thread per row, by descending degree inside a part, the same for the same mesh."""
import ctypes

import numpy as np
import pytest

from simkit_amd import _lib
from simkit_amd.mesh import tetrahedralized_grid


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _order(X, T, precision):
    order, ptr, n = np.empty(len(X), np.int32), np.empty(257, np.int32), ctypes.c_int()
    _lib.call("sk_part_order", _ptr(X), _ptr(T), len(X), len(T), precision, _ptr(order), ctypes.byref(n), _ptr(ptr))
    return order, ptr[:n.value + 1]


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 4), (9, 5, 11), (2, 60, 2), (31, 17, 23), (48, 48, 48)])
@pytest.mark.parametrize("precision", [_lib.SK_PREC_FP64, _lib.SK_PREC_MIXED])
@pytest.mark.parametrize("shuffled", [False, True])
def test_part_order(n, precision, shuffled):
    X, T = tetrahedralized_grid(*[k + 1 for k in n])
    rng = np.random.default_rng(0)
    if shuffled:
        p = rng.permutation(len(X))
        inv = np.argsort(p)
        X, T = X[p], inv[T]
    X, T = np.ascontiguousarray(X, float), np.ascontiguousarray(T, np.int32)
    order, ptr = _order(X, T, precision)
    assert np.array_equal(np.sort(order), np.arange(len(X)))
    assert ptr[0] == 0 and ptr[-1] == len(X) and 1 <= len(ptr) - 1 <= 256
    rows = np.diff(ptr)
    assert rows.min() >= 1 and rows.max() <= 512
    pairs = np.unique(np.repeat(T, 4, 1).astype(np.int64).ravel() * len(X) + np.tile(T, (1, 4)).ravel())
    deg = np.bincount(pairs // len(X), minlength=len(X))
    for a, b in zip(ptr[:-1], ptr[1:]):
        assert (np.diff(deg[order[a:b]]) <= 0).all()
    again, ptr2 = _order(X, T, precision)
    assert np.array_equal(order, again) and np.array_equal(ptr, ptr2)


def test_part_order_of_a_mesh_too_large_for_the_chip_and_of_a_bad_one():
    X, T = tetrahedralized_grid(53, 53, 53)  # 148,877 vertices: more than 256 workgroups of 512 threads
    X, T = np.ascontiguousarray(X, float), np.ascontiguousarray(T, np.int32)
    order, ptr = _order(X, T, _lib.SK_PREC_FP64)
    assert len(ptr) == 1 and np.array_equal(np.sort(order), np.arange(len(X)))
    T[0, 0] = len(X)
    with pytest.raises(Exception):
        _order(X, T, _lib.SK_PREC_FP64)
