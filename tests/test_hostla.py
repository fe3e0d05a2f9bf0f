"""The host's symmetric eigensolver on matrices near tridiagonal form, as the
projections of a converging restarted Lanczos run are: the entries outside
the band shrink towards nothing, and count as long as they are there."""
import ctypes as C

import numpy as np
import pytest

import dmed


@pytest.mark.parametrize("coupling", [1.0, 1e-4, 1e-8, 1e-9, 1e-12, 1e-17, 0.0])
@pytest.mark.parametrize("n", [2, 3, 8, 60])
def test_syev_near_tridiagonal(n, coupling):
    rng = np.random.default_rng(n)
    A = coupling * rng.uniform(0.5, 1, (n, n)) / n
    T = A + A.T + np.diag(rng.uniform(-4, 4, n)) + np.eye(n, k=1) + np.eye(n, k=-1)
    a, w = np.array(T, order="F"), np.zeros(n)
    f = getattr(dmed.lib(), "_ZN4dmed9host_syevEiPdS0_")
    assert f(C.c_int(n), a.ctypes.data_as(C.c_void_p), w.ctypes.data_as(C.c_void_p)) == 0
    # backward stable: a few ulp of ||T|| <= 8 per row
    tol = 8 * n * 2.0 ** -53 * 8
    assert np.abs(T @ a - a * w).max() <= tol
    assert np.abs(a.T @ a - np.eye(n)).max() <= tol
    assert np.abs(np.sort(w) - np.linalg.eigvalsh(T)).max() <= tol
