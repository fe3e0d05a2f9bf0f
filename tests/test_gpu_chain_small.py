"""The one-workgroup Lanczos chain of small sectors against plain Lanczos on
the oracle's H*v with reductions in extended precision, at the edges of its launch shapes: one row or one column, a row
for nearly every lane (1001), one to eight columns per lane, the largest
sector and the first one past it, spin exchange and pair hopping, both
precisions and the mixed form, an early exit and a zero start vector."""
import numpy as np
import pytest

import dmed
import edref

pytestmark = pytest.mark.gpu
NSTEP = 12


@pytest.fixture(scope="module", autouse=True)
def gpu():
    edref.build()
    dmed.init(0)
    yield


def model(norb, nbath, jh=0, seed=0):
    rng = np.random.default_rng(seed)
    bath = np.concatenate([rng.uniform(-1, 1, norb * nbath), rng.uniform(0.3, 0.6, norb * nbath)])
    hloc = np.diag(0.1 * np.arange(norb)).flatten(order="F")
    args = (norb, nbath, 1, bath, hloc, [2.0] * norb, 1.5, 0.25, 0.2 * jh, 0.15 * jh, 0.1, True, bool(jh))
    edref.set_model(*args)
    return dmed.set_model(*args)


def lanczos(m, x, n):
    """Plain Lanczos on the oracle's H*v; dot products, norms and vector
    updates in extended precision, so that its own sums add no error."""
    v = x.astype(np.longdouble)
    v, vp, b = v / np.sqrt(v @ v), np.zeros_like(v), np.longdouble(0)
    al, be = np.zeros(n), np.zeros(n)
    for k in range(n):
        w = edref.hxv(m, v.astype(np.float64)).real.astype(np.longdouble) - b * vp
        a = w @ v
        w = w - a * v
        b = np.sqrt(w @ w)
        al[k] = a
        if k + 1 < n:
            be[k + 1] = b
        if b < 1e-13:
            return al, be, k + 1
        vp, v = v, w / b
    return al, be, n


@pytest.mark.parametrize("norb,nbath,nup,ndw,jh", [
    (1, 7, 0, 4, 0), (1, 7, 4, 0, 0), (1, 5, 1, 1, 0), (1, 5, 3, 3, 0), (1, 7, 4, 3, 0), (1, 7, 4, 4, 0),
    (1, 8, 4, 2, 0), (1, 8, 3, 3, 0), (1, 11, 4, 1, 0), (1, 11, 1, 4, 0), (1, 13, 4, 0, 0), (1, 13, 0, 4, 0),
    (1, 11, 2, 2, 0), (1, 16, 2, 1, 0), (1, 8, 4, 3, 0), (2, 2, 3, 3, 1), (2, 3, 4, 4, 1), (3, 1, 3, 3, 1), (3, 2, 2, 4, 0)])
@pytest.mark.parametrize("prec", [dmed.FP64, dmed.FP32])
def test_small_chain_vs_oracle(norb, nbath, nup, ndw, jh, prec):
    print(f"[small chain] norb={norb} nbath={nbath} {nup}/{ndw} jh={jh} prec={prec}", flush=True)
    model(norb, nbath, jh)
    s = dmed.Sector(nup, ndw)
    x = np.random.default_rng(s.dim).standard_normal(s.dim)
    if prec == dmed.FP32:
        x = x.astype(np.float32).astype(np.float64)
    n = min(NSTEP, s.dim)
    a, b, ns = dmed.chain(s, s.vec(x, prec), n, prec=prec)
    ar, br, nr = lanczos(edref.build_sector(nup, ndw), x, n)
    assert ns == nr
    # a step adds a few roundings of ||H|| <= |a| + 2|b|, and the recurrence
    # carries them on: a factor of four a step bounds it while no Ritz value
    # has converged
    k = min(ns, 6 if prec == dmed.FP32 else NSTEP)
    u = 2.0 ** -24 if prec == dmed.FP32 else 2.0 ** -53
    tol = 4 * u * (np.abs(ar).max() + 2 * np.abs(br).max()) * 4.0 ** np.arange(k)
    assert (np.abs(a[:k] - ar[:k]) <= tol).all() and (np.abs(b[:k] - br[:k]) <= tol).all()


def test_small_chain_mixed_head_and_exits():
    ns = model(1, 7)
    s = dmed.Sector(4, 4)
    x = np.random.default_rng(1).standard_normal(s.dim)
    v = s.vec(x)
    a, b, n = dmed.chain(s, v, 60)
    am, bm, nm = dmed.chain(s, v, 60, prec=dmed.MIXED)
    assert n == nm == 60
    # the FP64 head of a mixed chain is the FP64 chain
    assert np.array_equal(a[:32], am[:32]) and np.array_equal(b[:32], bm[:32])
    assert np.abs(a[32:36] - am[32:36]).max() < 1e-4
    # the chain of an eigenvector ends after one step, of a zero vector at once
    ev, vecs, _, _ = s.eigh(1)
    a, b, n = dmed.chain(s, vecs[0], 20, threshold=1e-9)
    assert n == 1 and abs(a[0] - ev[0]) < 1e-10 and not a[1:].any() and not b[2:].any()
    a, b, n = dmed.chain(s, s.vec(np.zeros(s.dim)), 20)
    assert n == 0 and not a.any()
    # chains of the sector continue from nothing but their start vector
    a1, b1, _ = dmed.chain(s, v, 60)
    a2, b2, _ = dmed.chain(s, v, 60)
    assert np.array_equal(a1, a2) and np.array_equal(b1, b2)


@pytest.mark.parametrize("norb,nbath,nup,ndw,jh", [
    (1, 5, 3, 3, 0), (1, 7, 4, 3, 0), (1, 8, 3, 3, 0), (2, 3, 4, 4, 1), (1, 8, 4, 4, 0)])
@pytest.mark.parametrize("prec", [dmed.FP64, dmed.MIXED])
def test_small_ground_state(norb, nbath, nup, ndw, jh, prec):
    """The two-pass ground state, whose second pass adds up the vector: its
    residual is below the tolerance, on the oracle's H*v too."""
    print(f"[small ground] norb={norb} nbath={nbath} {nup}/{ndw} jh={jh} prec={prec}", flush=True)
    model(norb, nbath, jh)
    s = dmed.Sector(nup, ndw)
    e, v, res, rc = s.ground_state(prec=prec, tol=1e-11)
    assert rc == 0 and res <= 1e-11 * max(1, abs(e))
    x = v.download()
    w = edref.hxv(edref.build_sector(nup, ndw), x).real
    # 1e-11 asked for, plus the roundings of two H*v (a few ulp of ||H|| <= 60)
    assert np.linalg.norm(w - e * x) <= 1e-11 * max(1, abs(e)) + 1e-12
    assert abs(np.linalg.norm(x) - 1) < 1e-13
    ev, _, _, rc = s.eigh(1, dense_threshold=16)
    assert rc == 0 and abs(ev[0] - e) < 1e-10


@pytest.mark.parametrize("norb,nbath,jh,nst,chi", [(1, 7, 0, 1, 0), (1, 8, 0, 8, 0), (2, 3, 1, 6, 1), (2, 2, 0, 24, 1), (1, 3, 0, 4, 0)])
@pytest.mark.parametrize("batched", [0, 1])
def test_chain_batch_of_a_solve(norb, nbath, jh, nst, chi, batched):
    """The chains of a solve in one launch against the same chains one by one
    (the mixed form with every step in its FP64 head takes that way): one to
    eight columns per lane, stacked sectors beside plain ones, chains longer
    than their sector."""
    print(f"[chain batch] {norb} {nbath} jh={jh} nst={nst} chi={chi} batched={batched}", flush=True)
    ns = model(norb, nbath, jh)
    kw = dict(lanc_nstates_sector=2, lanc_nstates_total=nst, lmats=64, lreal=64, beta=20.0, eps=0.1,
              ltau=40, chi_spin=chi, chi_dens=chi, lanc_ngfiter=100, batched=batched)
    a = dmed.solve(norb, 1, ns, dmed.default_params(prec_gf=dmed.FP64, **kw))
    ns = model(norb, nbath, jh)
    b = dmed.solve(norb, 1, ns, dmed.default_params(prec_gf=dmed.MIXED, gf_fp64_head=100, **kw))
    assert a["nstates"] == b["nstates"] and abs(a["egs"] - b["egs"]) < 1e-10
    # the bars of the solve against the oracle on the same quantities
    keys = ["gmats"] + [k for k in a if chi and k.endswith(("chi_iv", "chi_tau"))]
    for k in keys:
        x, y = np.asarray(a[k]), np.asarray(b[k])
        assert np.abs(x - y).max() <= 1e-8 * max(1, np.abs(y).max()), k
