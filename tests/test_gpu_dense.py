"""Dense sectors on the device against numpy's eigen-decomposition of the
oracle's matrix: sizes around the host/device line, the row-group edges of the
1024-lane workgroup (512, 1024) and the largest size; spin exchange and pair
hopping; free and decoupled models with many equal levels; every eigenpair of
a sector; and the batch a solve launches, in both its forms."""
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


def model(norb, nbath, jh=0, u=2.0, v=0.4, seed=0):
    rng = np.random.default_rng(seed)
    bath = np.concatenate([rng.uniform(-1, 1, norb * nbath), v * rng.uniform(0.5, 1.0, norb * nbath)])
    args = (norb, nbath, 1, bath, np.zeros(norb * norb), [u] * norb, 0.75 * u, 0.1 * u, 0.1 * u * jh, 0.08 * u * jh,
            0.1, True, bool(jh))
    edref.set_model(*args)
    return dmed.set_model(*args)


@pytest.mark.parametrize("norb,nbath,nup,ndw,jh,u,v,neig", [
    (1, 7, 1, 1, 0, 2.0, 0.4, 6), (1, 5, 2, 1, 0, 2.0, 0.4, 3), (1, 5, 1, 1, 0, 2.0, 0.4, 36), (1, 5, 2, 2, 0, 2.0, 0.4, 6),
    (2, 2, 2, 3, 1, 2.0, 0.4, 6), (3, 1, 3, 3, 1, 2.0, 0.4, 12), (1, 5, 3, 3, 0, 0.0, 0.4, 9), (1, 5, 2, 3, 0, 2.0, 0.0, 9),
    (1, 7, 1, 4, 0, 2.0, 0.4, 4), (1, 6, 2, 3, 0, 2.0, 0.4, 4), (1, 13, 0, 4, 0, 2.0, 0.4, 17), (1, 9, 0, 5, 0, 2.0, 0.4, 2)])
def test_dense_sector_vs_numpy(norb, nbath, nup, ndw, jh, u, v, neig):
    print(f"[dense] norb={norb} nbath={nbath} {nup}/{ndw} jh={jh} u={u} v={v} neig={neig}", flush=True)
    model(norb, nbath, jh, u, v)
    s = dmed.Sector(nup, ndw)
    n = s.dim
    ev, vecs, res, rc = s.eigh(neig, dense_threshold=1024)
    assert rc == 0 and not res.any()
    H = edref.dense_h(edref.build_sector(nup, ndw)).real
    want = np.linalg.eigvalsh(H)
    # a backward-stable reduction and iteration move the levels by a small
    # multiple of n roundings of ||H||
    tol = 8 * n * U * max(np.abs(want).max(), 1.0)
    assert np.abs(ev - want[:neig]).max() <= tol
    X = np.array([x.download() for x in vecs])
    assert np.abs(X @ X.T - np.eye(neig)).max() <= 8 * n * U
    assert np.linalg.norm(X @ H - ev[:, None] * X, axis=1).max() <= 2 * tol
    e1, none, _, _ = s.eigh(neig, dense_threshold=1024, vectors=False)
    assert none is None and np.array_equal(e1, ev)


@pytest.mark.parametrize("finite", [0, 1])
def test_dense_batch_of_a_solve(finite):
    """Every sector of a small model dense: serial and batched solves launch
    the same batch, and agree with the solve whose larger sectors take the
    Krylov path."""
    ns = model(1, 4)
    kw = dict(beta=20.0, lmats=64, lreal=10, eps=0.3)
    if finite:
        kw.update(lanc_nstates_sector=6, lanc_nstates_total=30)
    print(f"[dense] solves, finite={finite}", flush=True)
    a, b, c = (dmed.solve(1, 1, ns, dmed.default_params(batched=bt, lanc_dim_threshold=th, **kw))
               for bt, th in ((0, 400), (1, 400), (0, 20)))
    for k in ("gmats", "greal", "smats", "dens"):
        assert np.array_equal(a[k], b[k]), k
    assert a["nstates"] == c["nstates"] and abs(a["egs"] - c["egs"]) < 1e-11
    assert np.abs(a["gmats"] - c["gmats"]).max() < 1e-9 and np.abs(a["dens"] - c["dens"]).max() < 1e-9
