"""H*v with spin exchange and pair hopping in the column kernel, long columns:
three to sixteen rows per lane (thirteen in FP64), a partial last row, and few
columns beside them, against the oracle, plain and in Lanczos mode, both
precisions."""
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


@pytest.mark.parametrize("norb,nbath,nup,ndw,bath_type", [
    (3, 4, 6, 2, "normal"), (3, 4, 7, 2, "normal"), (2, 7, 6, 2, "normal"), (2, 7, 7, 2, "normal"), (2, 7, 8, 2, "normal"),
    (3, 6, 4, 2, "normal"), (3, 5, 5, 2, "normal"), (2, 9, 5, 2, "normal"), (2, 12, 8, 12, "hybrid"), (2, 7, 8, 14, "normal")])
def test_long_columns_vs_oracle(norb, nbath, nup, ndw, bath_type):
    rng = np.random.default_rng(1)
    hyb = bath_type == "hybrid"
    bath = np.concatenate([rng.uniform(-1, 1, nbath if hyb else norb * nbath), rng.uniform(0.3, 0.6, norb * nbath)])
    hloc = np.diag(0.1 * np.arange(norb)).flatten(order="F")
    args = (norb, nbath, 1, bath, hloc, [2.0] * norb, 1.5, 0.25, 0.2, 0.15, 0.1, True, True)
    kw = dict(bath_type=bath_type) if hyb else {}
    edref.set_model(*args, **kw)
    dmed.set_model(*args, **kw)
    s = dmed.Sector(nup, ndw)
    rows = (s.dim_up + 1023) // 1024
    m = edref.build_sector(nup, ndw)
    x = rng.standard_normal(s.dim).astype(np.float32).astype(np.float64)
    ref = edref.hxv(m, x, nthreads=8).real
    for prec in (dmed.FP64, dmed.FP32):
        print(f"[col pairs long] norb={norb} nbath={nbath} {nup}/{ndw} {bath_type} prec={prec}", flush=True)
        assert s.hxv_shape(prec)["kernel"] == ("column" if rows <= 13 or prec == dmed.FP32 else "tile")
        # an element is a sum of at most 90 terms of |coefficient| <= 12, |x| < 7
        u = 2.0 ** -24 if prec == dmed.FP32 else 2.0 ** -53
        assert np.abs(s.hxv(x, prec) - ref).max() <= 90 * u * 90
        a, b, _ = dmed.chain(s, s.vec(x, prec), 2, prec=prec)
        assert abs(a[0] - x @ ref / (x @ x)) <= 100 * u * 30
