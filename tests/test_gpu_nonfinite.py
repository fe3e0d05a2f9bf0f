"""Models with NaN or infinite parameters, as a diverged bath fit leaves them:
the eigensolvers and the solve return (a NaN model's levels are NaN), reading
nothing out of bounds, and the next model is solved as if nothing had happened.  The dense
device solver's sectors (36 to 400 states) are among them, alone and in the
batch of a solve."""
import numpy as np
import pytest

import dmed

pytestmark = pytest.mark.gpu
NBATH = 5


@pytest.fixture(scope="module", autouse=True)
def gpu():
    dmed.init(0)
    yield


def model(**bad):
    rng = np.random.default_rng(3)
    bath = np.concatenate([rng.uniform(-1, 1, NBATH), rng.uniform(0.2, 0.5, NBATH)])
    u, xmu = 2.0, 0.0
    for k, x in bad.items():
        if k == "u":
            u = x
        elif k == "xmu":
            xmu = x
        else:
            bath[int(k[1:])] = x
    return dmed.set_model(1, NBATH, 1, bath, np.zeros(1), [u], 0.0, 0.0, 0.0, 0.0, xmu, True, False)


BAD = [dict(b1=np.nan), dict(b7=np.nan), dict(u=np.nan), dict(b0=np.inf), dict(b6=np.inf), dict(xmu=-np.inf)]


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("nup,ndw,neig", [(1, 1, 6), (2, 2, 6), (3, 3, 6), (2, 2, 225)])
def test_eigh(bad, nup, ndw, neig):
    print(f"[nonfinite] eigh {bad} {nup}/{ndw} neig={neig}", flush=True)
    model()
    s = dmed.Sector(nup, ndw)
    want = s.eigh(neig, dense_threshold=1024)[0]
    model(**bad)
    s = dmed.Sector(nup, ndw)
    try:
        ev, vecs, _, _ = s.eigh(neig, dense_threshold=1024)
        for v in vecs:
            v.download()
        if any(np.isnan(x) for x in bad.values()):
            assert not np.isfinite(ev).any()
    except dmed.DmedError as e:
        print(e, flush=True)
    model()
    s = dmed.Sector(nup, ndw)
    assert np.array_equal(s.eigh(neig, dense_threshold=1024)[0], want)


@pytest.mark.parametrize("bad", BAD)
@pytest.mark.parametrize("finite", [0, 1])
@pytest.mark.parametrize("batched", [0, 1])
def test_solve(bad, finite, batched):
    print(f"[nonfinite] solve {bad} finite={finite} batched={batched}", flush=True)
    kw = dict(beta=20.0, lmats=64, lreal=10, eps=0.3, batched=batched)
    if finite:
        kw.update(lanc_nstates_sector=6, lanc_nstates_total=30)
    p = dmed.default_params(**kw)
    ns = model()
    want = dmed.solve(1, 1, ns, p)
    ns = model(**bad)
    try:
        dmed.solve(1, 1, ns, p)
    except dmed.DmedError as e:
        print(e, flush=True)
    ns = model()
    got = dmed.solve(1, 1, ns, p)
    for k in ("egs", "gmats", "greal", "smats", "dens"):
        assert np.array_equal(got[k], want[k]), k
