"""The order in which the dense device solver takes its levels: a permutation
of the indices whatever the levels are, so that it can be used to index the
eigenvectors; ascending, equal levels by index, NaN last."""
import ctypes as C

import numpy as np
import pytest

import dmed


def order(d):
    d = np.ascontiguousarray(d, dtype=np.float64)
    o = np.full(len(d), -1, dtype=np.int32)
    f = getattr(dmed.lib(), "_ZN4dmed11dense_orderEiPKdPi")
    f.restype = None
    f(C.c_int(len(d)), d.ctypes.data_as(C.c_void_p), o.ctypes.data_as(C.c_void_p))
    return o


@pytest.mark.parametrize("n", [1, 2, 63, 225, 1024])
@pytest.mark.parametrize("kind", ["distinct", "equal", "some nan", "all nan", "infinite", "zeros"])
def test_order_is_a_permutation(n, kind):
    rng = np.random.default_rng(n)
    d = rng.standard_normal(n)
    if kind == "equal":
        d = np.round(d)
    elif kind == "some nan":
        d[rng.random(n) < 0.3] = np.nan
    elif kind == "all nan":
        d[:] = np.nan
    elif kind == "infinite":
        d[rng.random(n) < 0.2] = np.inf
        d[rng.random(n) < 0.2] = -np.inf
        d[n // 2] = -np.nan
    elif kind == "zeros":
        d = np.where(rng.random(n) < 0.5, 0.0, -0.0)
    o = order(d)
    assert np.array_equal(np.sort(o), np.arange(n))
    # numpy sorts stably, with NaN last
    assert np.array_equal(o, np.argsort(d, kind="stable"))
