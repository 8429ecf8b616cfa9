"""GPU: a batch that ends with an error gives its buffers back in order: the batches after it, which take them over,
and the operator's own solves give the bits that they gave before."""
import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.util import random_fermion

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver,sloppy", [(cmx.CG, cmx.DOUBLE), (cmx.RELIABLE_CG, cmx.HALF), (cmx.FGMRESDR, cmx.SINGLE)])
def test_after_an_error(solver, sloppy):
    L = (4, 6, 4, 8)
    Vh = int(np.prod(L)) // 2
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=2, eps=0.3), (1, 1, 1, -1))
    op = cmx.Operator(cmx.Gauge(L, U), cmx.EO_WILSON, cmx.kappa_to_mass(0.11), sloppy_prec=cmx.HALF)
    chis = [random_fermion(2 * Vh, 10 + k)[Vh:] for k in range(3)]
    kw = dict(solver=solver, rsd=1e-8, sloppy_prec=sloppy, tune=False)
    want = [p.tobytes() for p in cmx.solve_batch([op] * 3, chis, **kw)[0]]
    bad = [chis[0], np.full_like(chis[1], np.nan), chis[2]]
    raised = 0
    for src, maxit in ((chis, 2), (bad, 500), (chis, 5), (bad, 500)):
        print("batch error", solver, sloppy, maxit, flush=True)
        try:  # CG returns what it has at MaxIter, the other solvers raise
            cmx.solve_batch([op] * 3, src, maxit=maxit, **kw)
        except cmx.CmxError:
            raised += 1
        assert [p.tobytes() for p in cmx.solve_batch([op] * 3, chis, **kw)[0]] == want
    assert raised >= 2
