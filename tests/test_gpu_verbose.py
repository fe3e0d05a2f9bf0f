"""A verbose solve names every sector that it diagonalises, whichever solver
takes it: the dense batch, the sector queue or a worker."""
import os
import re
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dmft-ed_amd")

CHILD = """
import sys
import numpy as np
sys.path.insert(0, {pkg!r})
import dmed
dmed.init(0)
ns = dmed.set_model(1, 5, 2, np.concatenate([np.linspace(-1, 1, 10), np.full(10, 0.3)]), np.zeros((2, 2, 1, 1)), [2.0])
p = dmed.default_params(beta=20.0, lmats=16, lreal=4, eps=0.3, verbose=2, batched={batched}, lanc_nstates_sector=2,
                        lanc_nstates_total=6)
dmed.solve(1, 2, ns, p)
"""


@pytest.mark.parametrize("batched", [0, 1])
def test_every_sector_is_named(batched):
    print(f"[verbose] batched={batched}", flush=True)
    r = subprocess.run([sys.executable, "-u", "-c", CHILD.format(pkg=PKG, batched=batched)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert {int(k) for k in re.findall(r"^sector (\d+) dim=", r.stderr, re.M)} == set(range(49))
