"""GPU: failed captures of a Lanczos step graph, at every step of both captured
windows: six steps where a step is two launches (up to 2^22 states), three
where it is four (beyond).  The eager loop resumes from the vectors and the set
of scalars as they were before the capture: alpha and beta equal the all-eager
chain (DMED_GRAPHS=0) bit for bit, FP64 and mixed.  Each setting runs in a child
process, since both are read once per process."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dmft-ed_amd")

CHILD = r'''
import sys
import numpy as np
sys.path.insert(0, {pkg!r})
import dmed
dmed.init(0)
nbath, nup, ndw = {sector!r}
rng = np.random.default_rng(3)
dmed.set_model(1, nbath, 1, np.concatenate([rng.uniform(-1, 1, nbath), rng.uniform(0.2, 0.5, nbath)]), np.zeros(1), [2.0])
s = dmed.Sector(nup, ndw)
x = np.random.default_rng(21).standard_normal(s.dim)
out = {{"dim": s.dim}}
for name, prec in (("fp64", dmed.FP64), ("mixed", dmed.MIXED)):
    a, b, n = dmed.chain(s, s.vec(x), 70, prec=prec)
    out["a_" + name], out["b_" + name] = a, b
np.savez({out!r}, **out)
'''


def _child(tmp, sector, **env):
    out = os.path.join(tmp, "out.npz")
    print(f"[capture windows] {sector} {env}", flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", CHILD.format(pkg=PKG, sector=sector, out=out)],
                       env=dict(os.environ, DMED_TUNE="0", **env), capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return dict(np.load(out)), r.stderr


@pytest.mark.parametrize("sector,window,past", [((11, 5, 6), 6, False), ((13, 5, 6), 3, True)])
def test_failed_capture_at_every_step(tmp_path, sector, window, past):
    ref, _ = _child(str(tmp_path), sector, DMED_GRAPHS="0")
    assert (int(ref["dim"]) > 1 << 22) == past
    got, err = _child(str(tmp_path), sector)
    assert "capture unavailable" not in err
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k
    for q in range(window):
        got, err = _child(str(tmp_path), sector, DMED_TEST_CAPTURE_FAIL=str(q))
        assert "capture unavailable" in err
        for k in ref:
            assert np.array_equal(got[k], ref[k]), (q, k)
    _, err = _child(str(tmp_path), sector, DMED_TEST_CAPTURE_FAIL=str(window))
    assert "capture unavailable" not in err         # past the window: nothing fails
