"""GPU: a batched learned FGMRES-DR has its buffers before its timed region, not from the first step on (an allocation
there waits for the driver to clear memory that an earlier call released).  Zero sources make no step at all, so the
network's batch buffers, which stay with the operator, show whether they were there before one."""
import ctypes

import numpy as np
import pytest

from chroma_amd import lib as cmx

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so.7").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_network_buffers_before_the_first_step():
    L = (16, 16, 16, 32)
    Vh = int(np.prod(L)) // 2
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=2, eps=0.3), (1, 1, 1, -1))
    mass = cmx.kappa_to_mass(0.11)
    op = cmx.Operator(cmx.Gauge(L, U), cmx.EO_WILSON, mass, sloppy_prec=cmx.HALF)
    net = cmx.Net()
    net.init_neumann(4.0 + mass)
    cmx.net_attach(op, net)
    zero = np.zeros((Vh, 4, 3), complex)
    kw = dict(solver=cmx.FGMRESDR, rsd=1e-6, sloppy_prec=cmx.HALF, precond=cmx.PRECOND_LEARNED, n_krylov=4, tune=False)
    # the contexts' buffers, which stay in the scratch cache (1.2 GB)
    cmx.solve_batch([op] * 12, [zero] * 12, **dict(kw, precond=cmx.PRECOND_NONE))
    before = free_bytes()
    print("reserve", L, flush=True)
    _, res, summary = cmx.solve_batch([op] * 12, [zero] * 12, **kw)
    assert summary["n_iter"] == 0 and all(r["n_count"] == 0 for r in res)
    # a mixed field of 8 paths x 3 colours x 8 bytes per site and source
    assert before - free_bytes() >= 12 * 192 * Vh
