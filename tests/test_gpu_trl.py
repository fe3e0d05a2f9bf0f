"""Thick-restart Lanczos, whose expansion steps go in pairs, against dense
diagonalisation of the oracle's H: odd and even expansion lengths, the
smallest bases, sectors the basis spans, and Hamiltonians whose Krylov space
ends after a few steps (no hybridisation, equal bath levels), where the pairs
give way to single steps."""
import numpy as np
import pytest

import dmed
import edref

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    edref.build()
    dmed.init(0)
    yield


def model(norb, nbath, hyb, jh=0):
    rng = np.random.default_rng(7)
    eps = rng.uniform(-1, 1, norb * nbath) if hyb else np.zeros(norb * nbath)
    v = hyb * rng.uniform(0.3, 0.6, norb * nbath)
    hloc = np.diag(0.1 * np.arange(norb)).flatten(order="F")
    args = (norb, nbath, 1, np.concatenate([eps, v]), hloc, [2.0] * norb, 1.5, 0.25, 0.2 * jh,
            0.15 * jh, 0.1, True, bool(jh))
    edref.set_model(*args)
    return dmed.set_model(*args)


@pytest.mark.parametrize("norb,nbath,nup,ndw,jh", [(1, 5, 3, 3, 0), (1, 5, 2, 3, 0), (2, 2, 3, 3, 1), (1, 4, 1, 2, 0)])
@pytest.mark.parametrize("neig,ncv", [(1, 0), (1, 4), (2, 7), (3, 9), (4, 24)])
@pytest.mark.parametrize("hyb", [1.0, 1e-3, 0.0])
def test_trl_vs_dense(norb, nbath, nup, ndw, jh, neig, ncv, hyb):
    print(f"[trl] norb={norb} nbath={nbath} {nup}/{ndw} jh={jh} neig={neig} ncv={ncv} hyb={hyb}", flush=True)
    model(norb, nbath, hyb, jh)
    s = dmed.Sector(nup, ndw)
    ref = np.linalg.eigvalsh(edref.dense_h(edref.build_sector(nup, ndw)))
    ev, vecs, res, rc = s.eigh(neig, ncv=ncv, maxit=20000, tol=1e-11, dense_threshold=0)
    assert rc == 0
    # residuals below tol*max(1,|E|) give energies as close; |E| < 20
    assert np.abs(ev - ref[:neig]).max() <= 2e-10
    assert res.max() <= 1e-11 * max(1, np.abs(ev).max())
    X = np.array([v.download() for v in vecs])
    assert np.abs(X @ X.T - np.eye(neig)).max() < 1e-11
