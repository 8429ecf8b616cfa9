"""GPU: the launch shapes an operator has before any tuning, on lattices whose xy planes, z and t extents
fall on either side of the shapes' rules (planes of 2 to 288 sites, thin planes with more planes than
64-site groups, t extents with and without a factor 8), against the oracle at the storage precisions."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.test_gpu_parity import TOL
from tests.util import random_fermion, rel

pytestmark = pytest.mark.gpu

LATTICES = [(2, 2, 2, 2), (4, 4, 32, 30), (4, 2, 6, 8), (6, 10, 4, 10), (14, 10, 6, 6), (16, 18, 4, 8), (24, 24, 2, 4)]


@pytest.mark.parametrize("L", LATTICES)
@pytest.mark.parametrize("kind", [cmx.UNPREC_WILSON, cmx.EO_CLOVER])
def test_default_shapes(L, kind):
    V = int(np.prod(L))
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=5, eps=0.3), (1, 1, 1, -1))
    mass = cmx.kappa_to_mass(0.11)
    ref_op = oracle.Op(kind, L, U, mass, 1.0, 1.0)
    psi = random_fermion(V, 6)
    lo = 0 if kind == cmx.UNPREC_WILSON else V // 2
    for sloppy in (cmx.SINGLE, cmx.HALF):
        op = cmx.Operator(cmx.Gauge(L, U), kind, mass, 1.0, sloppy_prec=sloppy)
        for prec in (cmx.DOUBLE, sloppy):
            print("default shape", L, kind, prec, op.hop_config(prec), flush=True)
            assert op.hop_config(prec)["fast"] == 5  # all of these lattices are small enough for the direction-split kernel
            for isign in (+1, -1):
                assert rel(op(psi[lo:], isign, prec), ref_op(psi, isign)[lo:]) < TOL[prec]
        # |M p|^2 over every work-group: CG reaches its residual only with the right sums
        _, res = op.solve(psi[lo:], solver=cmx.CG, rsd=1e-10, maxit=500)
        assert res["rel_resid"] < 1e-8
