"""Which failures of a device path send a call to its host form: device memory
that cannot be had, and a pole iteration that did not converge; not an error
of the HIP runtime.  Device memory is asked for through exec_try, which leaves
no error behind for a later launch to report."""
import ctypes as C

import numpy as np
import pytest

import dmed

EHIP, ENOMEM, ENOCONV = -3, -4, -6


def _try(slot, nbytes):
    L = dmed.lib()
    ex = getattr(L, "_ZN4dmed2exEv")
    ex.restype = C.c_void_p
    f = getattr(L, "_ZN4dmed8exec_tryERNS_4ExecEimPPv")
    p = C.c_void_p()
    return f(C.c_void_p(ex()), C.c_int(slot), C.c_size_t(nbytes), C.byref(p)), p.value


@pytest.mark.parametrize("rc,host", [(0, False), (EHIP, False), (-1, False), (ENOMEM, True), (ENOCONV, True)])
def test_what_goes_to_the_host(rc, host):
    f = getattr(dmed.lib(), "_ZN4dmed13host_may_takeEi")
    f.restype = C.c_bool
    assert f(C.c_int(rc)) is host


@pytest.mark.gpu
def test_memory_that_cannot_be_had_leaves_nothing_behind():
    dmed.init(0)
    dmed.set_model(1, 3, 1, [-0.5, 0.1, 0.7, 0.3, 0.4, 0.2], np.zeros(1), [2.0])
    s = dmed.Sector(2, 2)
    x = np.random.default_rng(0).standard_normal(s.dim)
    want = s.hxv(x)
    assert _try(17, 1 << 50) == (ENOMEM, None)
    assert np.array_equal(s.hxv(x), want)           # the launch check sees no old error
    rc, p = _try(17, 1 << 12)
    assert rc == 0 and p


@pytest.mark.gpu
@pytest.mark.parametrize("slot", [11, 15, 16, 17])
def test_solve_without_room_for_a_buffer(slot, monkeypatch):
    """The solve's answers when one of its optional buffers cannot be had: the
    sums of G and chi (11), the dense sectors (15), the slab of start vectors
    (16) and the descriptors (17) of the chain batch."""
    dmed.init(0)
    rng = np.random.default_rng(4)
    bath = np.concatenate([rng.uniform(-1, 1, 5), rng.uniform(0.2, 0.5, 5)])
    ns = dmed.set_model(1, 5, 1, bath, np.zeros(1), [2.0])
    p = dmed.default_params(beta=20.0, lmats=64, lreal=10, eps=0.3, batched=1, chi_spin=1, chi_dens=1,
                            lanc_nstates_sector=4, lanc_nstates_total=20)
    want = dmed.solve(1, 1, ns, p)
    monkeypatch.setenv("DMED_TEST_NO_MEMORY", str(slot))
    print(f"[no memory] slot {slot}", flush=True)
    got = dmed.solve(1, 1, ns, p)
    # the same levels and chains to the solver's tolerance of 1e-12, in sums of
    # condition beta (chi) and 1/min |z| (G); orders of magnitude beyond it
    assert got["nstates"] == want["nstates"] and abs(got["egs"] - want["egs"]) < 1e-11
    for k, v in want.items():
        if isinstance(v, np.ndarray) and v.dtype.kind in "fc":
            assert np.abs(got[k] - v).max() <= 1e-8 * max(1.0, np.abs(v).max()), k
