"""The autotuner keeps its choices for sectors with spin exchange and pair
hopping apart from those of plain sectors of the same dimensions: one line
each in DMED_TUNE_FILE, either order of tuning, and the same H*v and chain
coefficients bit for bit as with the fixed rules.  In child processes, since
the settings are read once per process."""
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
rng = np.random.default_rng(1)
bath = np.concatenate([rng.uniform(-1, 1, 10), rng.uniform(0.3, 0.6, 10)])
out = {{}}
for jt in {order!r}:
    dmed.set_model(2, 5, 1, bath, np.zeros(4), [2.0, 2.0], 1.5, 0.25, 0.2 * jt, 0.15 * jt, 0.1, True, bool(jt))
    s = dmed.Sector(6, 3)
    x = np.random.default_rng(2).standard_normal(s.dim)
    out[f"y{{jt}}"] = s.hxv(x)
    a, b, n = dmed.chain(s, s.vec(x), 10)
    out[f"a{{jt}}"], out[f"b{{jt}}"] = a, b
np.savez({out!r}, **out)
'''


def _child(tmp, order, **env):
    out = os.path.join(tmp, "out.npz")
    print(f"[autotune pairs] order {order} {env}", flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", CHILD.format(pkg=PKG, order=order, out=out)],
                       env=dict(os.environ, **env), capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    return dict(np.load(out))


def test_pairs_have_choices_of_their_own(tmp_path):
    ref = _child(str(tmp_path), (0, 1), DMED_TUNE="0")
    for order in ((0, 1), (1, 0)):
        f = str(tmp_path / f"tune{order[0]}.txt")
        for _ in range(2):                      # tunes, then reads
            got = _child(str(tmp_path), order, DMED_TUNE="1", DMED_TUNE_MIN_DIM="0", DMED_TUNE_FILE=f)
            for k in ref:
                assert np.array_equal(got[k], ref[k]), (order, k)
        lines = [ln.split() for ln in open(f) if ln.strip()]
        assert sorted(int(ln[4]) for ln in lines) == [-4, 4]
