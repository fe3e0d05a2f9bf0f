"""Green's-function sums on the device (continued fractions) against the
pole sums of numpy's eigen-decomposition: chain lengths around the host/device
line and the largest, frequency counts around the block size, both isigns,
chains that ended early (zero-padded), and the forms that stay on the host
(a real axis without broadening)."""
import numpy as np
import pytest

import dmed
import edref

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.fixture(scope="module", autouse=True)
def gpu():
    edref.build()
    dmed.init(0)
    yield


def poles(a, b):
    lam, z = np.linalg.eigh(np.diag(a) + np.diag(b[1:], 1) + np.diag(b[1:], -1))
    return lam, z[0] ** 2


@pytest.mark.parametrize("n,lm,lr,isign,eps", [(15, 64, 3, 1, 0.05), (16, 63, 1, -1, 0.05), (17, 65, 0, 1, 0.05),
                                               (200, 1, 64, -1, 0.5), (301, 4097, 500, 1, 0.01), (1360, 0, 65, -1, 0.1),
                                               (40, 5, 7, 1, 0.0), (40, 5, 7, 1, -0.2)])
def test_gf_add_chain_vs_poles(n, lm, lr, isign, eps):
    print(f"[gf_sum] n={n} lm={lm} lr={lr} isign={isign} eps={eps}", flush=True)
    rng = np.random.default_rng(n + lm)
    a = rng.standard_normal(n)
    b = np.concatenate([[0.0], rng.uniform(0.3, 1.5, n - 1)])
    if n == 200:                                   # a chain that ended at step 120
        a[120:] = 0.0
        b[120] = 1e-14
        b[121:] = 0.0
    wm = np.pi / 40 * (2 * np.arange(lm) + 1)
    wr = np.linspace(-4.0, 4.0, lr) if lr > 1 else np.full(lr, 0.37)
    g0 = rng.standard_normal(lm) + 1j * rng.standard_normal(lm)
    r0 = rng.standard_normal(lr) + 1j * rng.standard_normal(lr)
    g, r = g0.copy(), r0.copy()
    dmed.gf_add_chain(0.7, -0.3, a, b, isign, wm, wr, eps, g, r)
    lam, w2 = poles(a, b)
    norm = np.abs(lam).max()
    for got, start, z in ((g, g0, 1j * wm), (r, r0, wr + 1j * eps)):
        if not len(z):
            continue
        want = start + (0.7 * w2 / (z[:, None] - isign * (lam - (-0.3)))).sum(1)
        # both sides see T to a few units of rounding: |dG| <= |dT| / dist(z, spectrum)^2
        dist = np.abs(z[:, None] - isign * (lam + 0.3)).min(1)
        tol = 0.7 * 40 * U * (norm + np.abs(z)) / dist ** 2 + 8 * U * (np.abs(start) + 0.7 / dist)
        assert (np.abs(got - want) <= tol).all(), (np.abs(got - want) / tol).max()


def test_many_states_solve_vs_oracle():
    """More chains per Green's function than one launch takes (64): every state
    of a small model kept at a high temperature, against the oracle's solve."""
    rng = np.random.default_rng(8)
    e, v = rng.uniform(-1, 1, 3), rng.uniform(0.3, 0.6, 3)
    bath, hloc = np.concatenate([e, v]), np.zeros(1)
    kw = dict(beta=1.0, lmats=70, lreal=20, eps=0.2, lanc_ngfiter=100, lanc_nstates_sector=36, lanc_nstates_total=256)
    print("[gf_sum] finite-temperature solve with all states", flush=True)
    ns = dmed.set_model(1, 3, 1, bath, hloc, [2.0])
    r = dmed.solve(1, 1, ns, dmed.default_params(**kw))
    assert 2 * r["nstates"] > 128
    o = edref.ed_solve(1, 3, 1, bath, hloc, [2.0], 0.0, 0.0, 0.0, True, params=edref.default_params(**kw))
    assert r["nstates"] == len(o["states"])
    assert np.abs(r["gmats"][0, 0, 0, 0] - o["gmats"][0, 0]).max() < 1e-10
    assert np.abs(r["smats"][0, 0, 0, 0] - o["smats"][0, 0]).max() < 1e-8


@pytest.mark.parametrize("n,nv,nt,lr,beta", [(15, 65, 64, 3, 20.0), (16, 1, 1, 1, 20.0), (17, 64, 0, 65, 5.0),
                                             (200, 0, 1001, 0, 50.0), (301, 1025, 129, 500, 50.0), (1360, 7, 5, 3, 10.0)])
def test_chi_add_chain_vs_poles(n, nv, nt, lr, beta):
    print(f"[chi_sum] n={n} nv={nv} nt={nt} lr={lr} beta={beta}", flush=True)
    rng = np.random.default_rng(n + nv)
    a = rng.uniform(-0.5, 0.5, n)
    b = np.concatenate([[0.0], rng.uniform(0.3, 1.2, n - 1)])
    if n == 200:                                   # a chain that ended at step 150
        a[150:] = 0.0
        b[150:] = 0.0
    ei = -2.0 * np.abs(b).max() - 1.0              # below the chain's levels
    vm = 2 * np.pi / beta * np.arange(nv)
    tau = np.linspace(0.0, beta, nt)
    wr, eps = np.linspace(-4.0, 4.0, lr), 0.1
    start = rng.standard_normal(nv) + 0j, rng.standard_normal(nt), rng.standard_normal(lr) + 0j
    iv, ct, cw = (x.copy() for x in start)
    dmed.chi_add_chain(0.7, 0.9, ei, a, b, beta, vm, tau, wr, eps, iv, ct, cw)
    lam, w2 = poles(a, b)
    de, w = lam - ei, 0.63 * w2
    num = np.exp(-beta * de) - 1.0
    f = np.where(beta * de < 0.1, beta, -num / de)

    def both(z):
        return (w * num / (z[:, None] - de) - w * num / (z[:, None] + de)).sum(1)

    want = [start[0] + (both(1j * vm) if nv else 0), start[1] + 0.0, start[2] + (both(wr + 1j * eps) if lr else 0)]
    if nv:
        want[0][0] = start[0][0] + 2 * (w * f).sum()
    if nt:
        want[1] = start[1] + (w * (np.exp(-tau[:, None] * de) + np.exp(-(beta - tau)[:, None] * de))).sum(1)
    # errors of the levels of a few units of rounding of ||T||, amplified by
    # beta in the exponentials and by the squared distance to the poles
    u = 60 * U * (np.abs(lam).max() + abs(ei))
    assert (np.abs(iv - want[0]) <= 0.63 * u * 4 / de.min() ** 2 + 16 * U * np.abs(want[0])).all() if nv else True
    assert (np.abs(ct - want[1]) <= 0.63 * u * 2 * beta + 16 * U * (1 + np.abs(want[1]))).all() if nt else True
    assert (np.abs(cw - want[2]) <= 0.63 * u * 4 / eps ** 2 + 16 * U * np.abs(want[2])).all() if lr else True
