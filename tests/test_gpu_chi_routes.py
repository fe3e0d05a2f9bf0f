"""Susceptibilities of solves with enough chains for the device to find their
poles too (one wave a chain, 1 to 36 steps and 65 to 200), and with few, whose
poles the host finds on its threads, against the sums on the host alone (taken
where the device buffer cannot be had); and a single chain at the lines
between the forms, which adds to what is there."""
import numpy as np
import pytest

import dmed

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    dmed.init(0)
    yield


@pytest.mark.parametrize("norb,nbath,nsec,ntot,ngf,beta", [
    (2, 1, 36, 256, 200, 2.0), (2, 3, 4, 20, 200, 20.0), (2, 3, 4, 20, 65, 20.0), (1, 5, 2, 4, 200, 20.0),
    (1, 5, 1, 1, 200, 20.0)])
@pytest.mark.parametrize("batched", [0, 1])
def test_solve(norb, nbath, nsec, ntot, ngf, beta, batched, monkeypatch):
    print(f"[chi routes] {norb}x{nbath} {ntot} states, {ngf} steps, batched={batched}", flush=True)
    rng = np.random.default_rng(6)
    n = norb * nbath
    bath = np.concatenate([rng.uniform(-1, 1, n), rng.uniform(0.2, 0.5, n)])
    ns = dmed.set_model(norb, nbath, 1, bath, np.zeros(norb * norb), [2.0] * norb, 1.5, 0.25)
    p = dmed.default_params(beta=beta, lmats=200, lreal=50, eps=0.3, batched=batched, chi_spin=1, chi_dens=1,
                            lanc_nstates_sector=nsec, lanc_nstates_total=ntot, lanc_ngfiter=ngf)
    got = dmed.solve(norb, 1, ns, p)
    monkeypatch.setenv("DMED_TEST_NO_MEMORY", "11")
    want = dmed.solve(norb, 1, ns, p)
    # levels within 60 units of rounding of ||T|| + |E| <= 20, twice; at most
    # beta^2 or 4/eps^2 in the sums, with weights of at most 4 a state
    tol = 2 * 60 * 2.0 ** -53 * 20 * max(beta ** 2, 4 / 0.3 ** 2) * 4
    keys = [k for k in want if "chi" in k]
    assert len(keys) == 12
    for k in keys:
        assert np.abs(got[k] - want[k]).max() <= tol + 1e-13 * np.abs(want[k]).max(), k


@pytest.mark.parametrize("n", [1, 2, 10, 24, 26, 28, 60, 95])
@pytest.mark.parametrize("nv,nt,lr", [(33, 21, 50), (1025, 101, 500), (0, 0, 1)])
def test_one_chain(n, nv, nt, lr, monkeypatch):
    rng = np.random.default_rng(n)
    a, b = rng.uniform(-0.5, 0.5, n), np.concatenate([[0.0], rng.uniform(0.3, 1.2, n - 1)])
    vm, tau, wr = 2 * np.pi / 20 * np.arange(nv), np.linspace(0, 20.0, nt), np.linspace(-4, 4, lr)
    wm = np.pi / 20 * (2 * np.arange(nv) + 1)

    def run():
        iv, ct, cw = np.ones(nv, complex), np.ones(nt), np.ones(lr, complex)
        dmed.chi_add_chain(0.7, 0.9, -4.0, a, b, 20.0, vm, tau, wr, 0.3, iv, ct, cw)
        gm, gr = np.ones(nv, complex), np.ones(lr, complex)
        dmed.gf_add_chain(0.7, -4.0, a, b, 1, wm, wr, 0.3, gm, gr)
        return iv, ct, cw, gm, gr

    print(f"[chi routes] n={n} {nv}/{nt}/{lr}", flush=True)
    got = run()
    monkeypatch.setenv("DMED_TEST_NO_MEMORY", "11")
    tol = 2 * 60 * 2.0 ** -53 * 10 * 400            # as above
    for x, y in zip(got, run()):
        assert x.shape == y.shape and (np.abs(x - y) <= tol).all()
