"""Thick-restart Lanczos where the Krylov space of a start vector ends inside
the first cycle (equal bath levels with hybridisation: few distinct
energies), so that the steps before the end stand and the rest are taken
again: levels with their multiplicities, residuals and orthogonality against
dense diagonalisation of the oracle's H."""
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


@pytest.mark.parametrize("norb,nbath,nup,ndw", [(1, 5, 3, 3), (1, 6, 3, 3), (1, 5, 2, 3), (2, 2, 3, 3)])
@pytest.mark.parametrize("neig,ncv", [(1, 0), (1, 7), (1, 40), (3, 9), (6, 24), (6, 0)])
def test_equal_levels(norb, nbath, nup, ndw, neig, ncv):
    print(f"[trl short] {norb}x{nbath} {nup}/{ndw} neig={neig} ncv={ncv}", flush=True)
    rng = np.random.default_rng(5)
    n = norb * nbath
    args = (norb, nbath, 1, np.concatenate([np.zeros(n), rng.uniform(0.2, 0.5, n)]),
            np.zeros(norb * norb), [2.0] * norb, 1.5, 0.25, 0.0, 0.0, 0.1, True, False)
    edref.set_model(*args)
    dmed.set_model(*args)
    s = dmed.Sector(nup, ndw)
    ref = np.linalg.eigvalsh(edref.dense_h(edref.build_sector(nup, ndw)))
    ev, vecs, res, rc = s.eigh(neig, ncv=ncv, maxit=20000, tol=1e-11, dense_threshold=0)
    assert rc == 0
    # residuals below tol*max(1,|E|) give energies as close; |E| < 20
    assert np.abs(ev - ref[:neig]).max() <= 2e-10
    assert res.max() <= 1e-11 * max(1, np.abs(ev).max())
    X = np.array([v.download() for v in vecs])
    assert np.abs(X @ X.T - np.eye(neig)).max() < 1e-11
