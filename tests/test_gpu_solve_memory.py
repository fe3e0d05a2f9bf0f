"""Device memory that repeated solves hold: the work space of the dense batch
(here about 40 MB) stays in one execution context, whichever contexts the
workers of the solves take between."""
import ctypes as C

import numpy as np
import pytest

import dmed

pytestmark = pytest.mark.gpu


def _free_bytes():
    hip = C.CDLL("libamdhip64.so")
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def test_repeated_solves_hold_one_dense_work_space():
    dmed.init(0)
    rng = np.random.default_rng(2)
    bath = np.concatenate([rng.uniform(-1, 1, 6), rng.uniform(0.2, 0.5, 6)])
    ns = dmed.set_model(1, 6, 1, bath, np.zeros(1), [2.0])
    p = dmed.default_params(beta=20.0, lmats=64, lreal=10, eps=0.3, batched=1, lanc_dim_threshold=1024,
                            lanc_nstates_sector=2, lanc_nstates_total=6)
    left = []
    for i in range(8):
        dmed.solve(1, 1, ns, p)
        left.append(_free_bytes())
        print(f"[solve memory] after solve {i}: {left[-1] >> 20} MB free", flush=True)
    # the workers' own buffers may still grow by a few MB
    assert left[0] - left[-1] < 20 << 20
