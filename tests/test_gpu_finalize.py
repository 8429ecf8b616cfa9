"""GPU: reductions of 4, 576 and 2592 partials, on both sides of the size where the finishing group grows, alone and
in one batch whose group has the size of the largest: the same bits, and the residual that the solver claims."""
import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.util import random_fermion

pytestmark = pytest.mark.gpu

LATTICES = [(4, 4, 4, 8), (16, 16, 16, 18), (24, 24, 24, 24)]


@pytest.mark.parametrize("solver", [cmx.CG, cmx.RELIABLE_CG])
def test_sizes(solver):
    ops, chis, single = [], [], []
    for L in LATTICES:
        print("finalize", L, solver, flush=True)
        U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=4, eps=0.3), (1, 1, 1, -1))
        op = cmx.Operator(cmx.Gauge(L, U), cmx.EO_WILSON, cmx.kappa_to_mass(0.11))
        chi = random_fermion(int(np.prod(L)), 3)[int(np.prod(L)) // 2:]
        psi, res = op.solve(chi, solver=solver, rsd=1e-9, sloppy_prec=cmx.SINGLE)
        # |chi - M psi| <= |M^-dag| |M^dag chi - M^dag M psi|, and |M| |M^-1| < 30 at this kappa
        assert res["rel_resid"] < 30 * 1e-9
        ops.append(op), chis.append(chi), single.append(psi)
    psis, _, _ = cmx.solve_batch(ops, chis, solver=solver, rsd=1e-9, sloppy_prec=cmx.SINGLE, tune=False)
    assert [p.tobytes() for p in psis] == [p.tobytes() for p in single]
