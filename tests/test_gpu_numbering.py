"""The vertex numbering follows the path the solves take: boxes or aggregates in index order for the resident PCG, the
sliced-ELL order (two-level: within each aggregate) for launches, which store their rows contiguously in it."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_resident import _box  # noqa: E402


def _order(entry, T, nv, *args):
    from simkit_amd import _lib
    order = np.empty(nv, np.int32)
    p = [a.ctypes.data_as(ctypes.c_void_p) if isinstance(a, np.ndarray) else a for a in args]
    Tc = np.ascontiguousarray(T, np.int32)
    if entry == "sk_sell_order":
        _lib.call(entry, Tc.ctypes.data_as(ctypes.c_void_p), nv, len(T), order.ctypes.data_as(ctypes.c_void_p))
        return order
    n, ptr = ctypes.c_int(), np.empty(nv + 1, np.int32)
    _lib.call(entry, p[0], nv, p[1], order.ctypes.data_as(ctypes.c_void_p), ctypes.byref(n),
              ptr.ctypes.data_as(ctypes.c_void_p))
    return order, ptr[:n.value + 1]


LAUNCHES = [{"pcg_chunk": 8}, {"spmv_blocks": 256}, {"update_blocks": 64}, {"pcg": "pipelined"}]


def _sim(n, **kw):
    from simkit_amd.sim import BackwardEulerSim
    X, T, fixed = _box(n, 3)
    return X, T, BackwardEulerSim(X, T, 3e5, 2e6, fixed_vertices=fixed, **kw)


@pytest.mark.parametrize("kw", LAUNCHES)
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_block_jacobi_launches_use_the_sliced_order(kw, precision):
    X, T, sim = _sim((9, 7, 8), precision=precision, **kw)
    sell = _order("sk_sell_order", T, len(X))
    resident = precision == "mixed" and "pcg" in kw  # mixed solves are classic whatever the variant
    assert np.array_equal(sim._order, sell) == (not resident)
    assert not np.array_equal(_sim((9, 7, 8), precision=precision)[2]._order, sell)


@pytest.mark.parametrize("n,kw", [((9, 7, 8), k) for k in LAUNCHES[:3]] + [((9, 7, 8), {}), ((52, 52, 52), {})])
def test_two_level_launches_use_the_sliced_order_within_aggregates(n, kw):
    X, T, sim = _sim(n, preconditioner="two_level", **kw)
    rank = np.empty(len(X), np.int64)
    rank[_order("sk_sell_order", T, len(X))] = np.arange(len(X))
    order, ptr = _order("sk_coarse_order", T, len(X), np.ascontiguousarray(X), sim.coarse_vertices)
    got = np.arange(len(X)) if sim._order is None else sim._order
    launches = bool(kw) or len(X) > 256 * 512
    for a, b in zip(ptr[:-1], ptr[1:]):
        want = order[a:b][np.argsort(rank[order[a:b]])] if launches else order[a:b]
        assert np.array_equal(got[a:b], want)
