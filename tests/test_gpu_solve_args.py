"""A solve that asks a sector for no eigenpair is refused before any work, also
where its sectors are all small enough for the dense batch."""
import numpy as np
import pytest

import dmed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [0, -2])
@pytest.mark.parametrize("total", [1, 10])
@pytest.mark.parametrize("batched", [0, 1])
def test_no_eigenpair_is_refused(count, total, batched):
    dmed.init(0)
    ns = dmed.set_model(1, 2, 1, [-0.5, 0.7, 0.3, 0.4], np.zeros(1), [2.0])
    kw = dict(beta=20.0, lmats=16, lreal=4, eps=0.3, batched=batched, lanc_nstates_total=total)
    want = dmed.solve(1, 1, ns, dmed.default_params(**kw))
    print(f"[solve args] lanc_nstates_sector={count}", flush=True)
    with pytest.raises(dmed.DmedError) as e:
        dmed.solve(1, 1, ns, dmed.default_params(lanc_nstates_sector=count, **kw))
    assert e.value.code == -1 and "neig" in str(e.value)
    got = dmed.solve(1, 1, ns, dmed.default_params(**kw))
    assert got["egs"] == want["egs"] and np.array_equal(got["gmats"], want["gmats"])
