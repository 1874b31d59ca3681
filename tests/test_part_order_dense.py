"""sk_part_order on a mesh with more blocks than the resident PCG's threads can hold: the launches' order (host only)."""
import ctypes

import numpy as np
import pytest

from simkit_amd import _lib


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.mark.parametrize("precision", [_lib.SK_PREC_FP64, _lib.SK_PREC_MIXED])
@pytest.mark.parametrize("per_vertex,dense", [(2, False), (12, True)])
def test_part_order_of_a_dense_mesh(precision, per_vertex, dense):
    nv = 50000  # random tets: 24 and 128 blocks a row, 9 and 49 for each of 256 x 512 threads on average
    rng = np.random.default_rng(1)
    X = rng.random((nv, 3))
    near = np.argsort(X[:, 0])
    T = near[(rng.integers(0, nv, (per_vertex * nv, 1)) + rng.integers(0, 400, (per_vertex * nv, 4))) % nv]
    T = np.ascontiguousarray(T, np.int32)
    order, sell, ptr, n = np.empty(nv, np.int32), np.empty(nv, np.int32), np.empty(257, np.int32), ctypes.c_int()
    _lib.call("sk_part_order", _ptr(X), _ptr(T), nv, len(T), precision, _ptr(order), ctypes.byref(n), _ptr(ptr))
    _lib.call("sk_sell_order", _ptr(T), nv, len(T), _ptr(sell))
    assert np.array_equal(np.sort(order), np.arange(nv))
    assert (n.value == 0) == dense and np.array_equal(order, sell) == dense
