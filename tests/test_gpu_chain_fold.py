"""The two-launch Lanczos step (sectors too large for one workgroup, up to 2^22
states) against plain Lanczos on the oracle's H*v with reductions in extended
precision, with the tile and the column kernel; chain lengths around the
captured window of six steps; an early end, a zero start vector, a restart."""
import numpy as np
import pytest

import dmed
import edref
from test_gpu_chain_small import lanczos, model

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    edref.build()
    dmed.init(0)
    yield


@pytest.mark.parametrize("norb,nbath,nup,ndw,jh", [(1, 8, 4, 4, 0), (1, 10, 5, 4, 0), (1, 11, 6, 3, 0), (1, 12, 5, 2, 0),
                                                   (2, 4, 4, 5, 1), (3, 3, 6, 2, 1)])
@pytest.mark.parametrize("prec", [dmed.FP64, dmed.FP32])
def test_fold_vs_oracle(norb, nbath, nup, ndw, jh, prec):
    print(f"[fold] norb={norb} nbath={nbath} {nup}/{ndw} jh={jh} prec={prec}", flush=True)
    model(norb, nbath, jh)
    s = dmed.Sector(nup, ndw)
    assert 8192 < s.dim <= 1 << 22
    x = np.random.default_rng(s.dim).standard_normal(s.dim)
    if prec == dmed.FP32:
        x = x.astype(np.float32).astype(np.float64)
    a, b, ns = dmed.chain(s, s.vec(x, prec), 12, prec=prec)
    ar, br, nr = lanczos(edref.build_sector(nup, ndw), x, 12)
    assert ns == nr
    # the bound of the one-workgroup chain's test
    k = min(ns, 6 if prec == dmed.FP32 else 12)
    u = 2.0 ** -24 if prec == dmed.FP32 else 2.0 ** -53
    tol = 4 * u * (np.abs(ar).max() + 2 * np.abs(br).max()) * 4.0 ** np.arange(k)
    assert (np.abs(a[:k] - ar[:k]) <= tol).all() and (np.abs(b[:k] - br[:k]) <= tol).all()


@pytest.mark.parametrize("prec", [dmed.FP64, dmed.FP32, dmed.MIXED])
def test_fold_lengths_and_ends(prec):
    print(f"[fold] lengths prec={prec}", flush=True)
    model(1, 8)
    s = dmed.Sector(4, 4)
    x = np.random.default_rng(2).standard_normal(s.dim)
    v = s.vec(x)
    a, b, n = dmed.chain(s, v, 100, prec=prec)
    assert n == 100
    # eager, one window, several windows and remainders: the same steps
    for m in (1, 2, 29, 30, 31, 36, 37, 42, 43, 67, 68, 69, 99):
        am, bm, nm = dmed.chain(s, v, m, prec=prec)
        assert nm == m and np.array_equal(am, a[:m]) and np.array_equal(bm, b[:m])
    if prec == dmed.FP64:
        ev, vecs, _, _ = s.eigh(1)
        for m in (20, 60):
            am, bm, nm = dmed.chain(s, vecs[0], m, threshold=1e-9)
            assert nm == 1 and abs(am[0] - ev[0]) < 1e-10 and not am[1:].any() and not bm[2:].any()
    am, bm, nm = dmed.chain(s, s.vec(np.zeros(s.dim)), 40, prec=prec)
    assert nm == 0 and not am.any()
    am, bm, nm = dmed.chain(s, v, 100, prec=prec)
    assert np.array_equal(am, a) and np.array_equal(bm, b)
