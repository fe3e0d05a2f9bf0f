"""H*v with spin exchange and pair hopping in the column kernel (D_up >= 512)
against the oracle, plain and in Lanczos mode, both precisions, one to four
rows per lane and a partial last row; and the sectors beside the rule's line,
which stay with the tile kernel."""
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


@pytest.mark.parametrize("norb,nbath,nup,ndw,kernel", [
    (3, 3, 6, 6, 2), (3, 3, 5, 3, 2), (3, 3, 7, 2, 2), (2, 5, 6, 3, 2), (2, 6, 6, 2, 2), (2, 6, 7, 12, 2), (2, 6, 7, 13, 1),
    (3, 3, 4, 6, 1), (2, 5, 6, 1, 1)])
@pytest.mark.parametrize("jx,jp", [(0.2, 0.15), (0.0, 0.3), (0.25, 0.0)])
@pytest.mark.parametrize("prec", [dmed.FP64, dmed.FP32])
def test_col_pairs_vs_oracle(norb, nbath, nup, ndw, kernel, jx, jp, prec):
    print(f"[col pairs] norb={norb} nbath={nbath} {nup}/{ndw} jx={jx} jp={jp} prec={prec}", flush=True)
    rng = np.random.default_rng(1)
    bath = np.concatenate([rng.uniform(-1, 1, norb * nbath), rng.uniform(0.3, 0.6, norb * nbath)])
    hloc = np.diag(0.1 * np.arange(norb)).flatten(order="F")
    args = (norb, nbath, 1, bath, hloc, [2.0] * norb, 1.5, 0.25, jx, jp, 0.1, True, True)
    edref.set_model(*args)
    dmed.set_model(*args)
    s = dmed.Sector(nup, ndw)
    assert s.hxv_shape(prec)["kernel"] == ("column" if kernel == 2 else "tile")
    m = edref.build_sector(nup, ndw)
    x = rng.standard_normal(s.dim)
    if prec == dmed.FP32:
        x = x.astype(np.float32).astype(np.float64)
    ref = edref.hxv(m, x, nthreads=8).real
    y, v = s.hxv(x, prec), s.vec(x, prec)
    # an element is a sum of at most 60 terms of |coefficient| <= 10, |x| < 6
    u = 2.0 ** -24 if prec == dmed.FP32 else 2.0 ** -53
    assert np.abs(y - ref).max() <= 60 * u * 60
    a, b, _ = dmed.chain(s, v, 2, prec=prec)
    n = np.linalg.norm(x)
    assert abs(a[0] - x @ ref / n ** 2) <= 100 * u * 20
