"""The host's symmetric eigensolver ends on infinite entries, wherever they
are."""
import ctypes as C

import numpy as np
import pytest

import dmed


@pytest.mark.parametrize("n", [2, 3, 4, 8])
@pytest.mark.parametrize("diagonal,coupling", [(np.inf, np.inf), (-np.inf, np.inf), (np.inf, 1.0), (1.0, np.inf)])
def test_syev_ends_on_infinite_entries(n, diagonal, coupling):
    for at in range(n - 1):
        A = np.asfortranarray(np.eye(n) + np.eye(n, k=1) + np.eye(n, k=-1))
        A[at, at + 1] = A[at + 1, at] = coupling
        A[at + 1, at + 1] = diagonal
        w = np.zeros(n)
        f = getattr(dmed.lib(), "_ZN4dmed9host_syevEiPdS0_")
        rc = f(C.c_int(n), A.ctypes.data_as(C.c_void_p), w.ctypes.data_as(C.c_void_p))
        assert rc in (0, -6)
