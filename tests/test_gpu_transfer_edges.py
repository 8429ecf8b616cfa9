"""GPU: what surrounds the staged transfers and the scratch cache.  Host arrays that are pinned already (copied without
staging), a cache that is full (its oldest buffers go, it stays below its 4 GiB), and calls after cmx_finalize has given
everything back; and the two ways in which a reliable solver's host reads the flags, bit for bit."""
import ctypes

import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.util import random_fermion

pytestmark = pytest.mark.gpu


def make_op(L):
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=2, eps=0.3), (1, 1, 1, -1))
    return cmx.Operator(cmx.Gauge(L, U), cmx.EO_WILSON, cmx.kappa_to_mass(0.11), sloppy_prec=cmx.HALF)


def hip():
    return ctypes.CDLL("libamdhip64.so.7")


@pytest.mark.parametrize("L", [(4, 4, 4, 8), (12, 12, 16, 20)])
def test_pinned_arrays(L):
    n = int(np.prod(L)) // 2
    op = make_op(L)
    x = random_fermion(2 * n, 4)[n:]
    want = op(x)
    h = hip()
    p = (ctypes.c_void_p(), ctypes.c_void_p())
    try:
        a = []
        for q in p:
            assert h.hipHostMalloc(ctypes.byref(q), ctypes.c_size_t(x.nbytes), 0) == 0
            a.append(np.frombuffer((ctypes.c_char * x.nbytes).from_address(q.value), np.complex128).reshape(x.shape))
        print("pinned", L, flush=True)
        a[0][...] = x
        dp = ctypes.POINTER(ctypes.c_double)
        cmx.check(cmx.lib().cmx_op_apply(op.h, a[1].ctypes.data_as(dp), a[0].ctypes.data_as(dp), 1, cmx.DOUBLE))
        assert a[1].tobytes() == want.tobytes()
    finally:
        for q in p:
            if q.value:
                h.hipHostFree(q)


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_full_cache_and_release():
    L = (4, 6, 4, 8)
    n = int(np.prod(L)) // 2
    op = make_op(L)
    x = random_fermion(2 * n, 4)[n:]
    want = op(x).tobytes()
    assert cmx.lib().cmx_finalize() == 0 and cmx.lib().cmx_init(0) == 0
    assert op(x).tobytes() == want
    before = free_bytes()
    for lt in (16, 24, 32, 44):  # two buffers of 0.30, 0.45, 0.60 and 0.83 GB: 4.4 GB in all
        dims = (32, 32, 32, lt)
        print("cache", dims, flush=True)
        U = np.zeros((4, int(np.prod(dims)), 3, 3), np.complex128)
        for c in range(3):
            U[..., c, c] = 1
        assert np.abs(cmx.gauge_stout_smear(dims, U, 1, 0.1) - U).max() < 1e-14
    assert op(x).tobytes() == want
    held = before - free_bytes()
    assert (3 << 30) < held <= (4 << 30) + (64 << 20), held
    assert cmx.lib().cmx_finalize() == 0 and cmx.lib().cmx_init(0) == 0
    assert before - free_bytes() < 64 << 20
    assert op(x).tobytes() == want


@pytest.mark.parametrize("solver,sloppy", [(cmx.RELIABLE_CG, cmx.HALF), (cmx.RELIABLE_CG, cmx.SINGLE),
                                           (cmx.RELIABLE_BICGSTAB, cmx.SINGLE)])
@pytest.mark.parametrize("delta", [0.5, 0.1])
def test_flags_read_ahead_or_not(solver, sloppy, delta):
    """verbose reads the flags after every iteration, small lattices otherwise one iteration behind the launches."""
    L = (4, 6, 4, 8)
    n = int(np.prod(L)) // 2
    op = make_op(L)
    x = random_fermion(2 * n, 4)[n:]
    kw = dict(solver=solver, rsd=1e-9, sloppy_prec=sloppy, delta=delta)
    a, ra = op.solve(x, **kw)
    b, rb = op.solve(x, verbose=True, **kw)
    print("ahead", solver, sloppy, delta, ra["n_count"], ra["n_reliable"], flush=True)
    assert a.tobytes() == b.tobytes()
    assert (ra["n_count"], ra["n_reliable"]) == (rb["n_count"], rb["n_reliable"]) and ra["n_reliable"] > 0
