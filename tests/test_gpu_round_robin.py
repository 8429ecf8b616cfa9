"""GPU: the plane-grid kernel with its planes handed out round-robin, on lattices of few and large time slices (the FP64
operator from 20000 sites per checkerboard and slice on, everything from 40000 on), whose xy planes fill the work-groups
or leave a ninth of the last one idle, against the oracle; and the reductions over that order."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.test_gpu_parity import TOL
from tests.util import random_fermion, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(36, 36, 36, 2), (48, 48, 48, 2), (20, 64, 64, 4)])
def test_round_robin(L):
    V = int(np.prod(L))
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=5, eps=0.3), (1, 1, 1, -1))
    mass = cmx.kappa_to_mass(0.11)
    op = cmx.Operator(cmx.Gauge(L, U), cmx.EO_CLOVER, mass, 1.0, sloppy_prec=cmx.HALF)
    assert op.hop_config(cmx.HALF)["fast"] == 1  # plane-grid by itself
    ref_op = oracle.Op(oracle.EO_CLOVER, L, U, mass, 1.0, 1.0)
    psi = random_fermion(V, 6)
    hop = oracle.dslash(L, U, psi, +1, 1)[V // 2:]
    ref = [ref_op(psi, isign)[V // 2:] for isign in (+1, -1)]
    for prec, fast in ((cmx.DOUBLE, 1), (cmx.DOUBLE, 3), (cmx.HALF, None), (cmx.SINGLE, 3)):
        for block in (64, 256):
            if fast is not None:
                op.set_hop_config(prec, block, 0, 1, 0, fast)
            print("round robin", L, prec, op.hop_config(prec), flush=True)
            for k, isign in enumerate((+1, -1)):
                assert rel(op(psi[V // 2:], isign, prec), ref[k]) < TOL[prec]
            assert rel(op.dslash(psi[: V // 2], +1, 1, prec), hop) < TOL[prec]
    _, res = op.solve(psi[V // 2:], solver=cmx.RELIABLE_CG, rsd=1e-10, sloppy_prec=cmx.HALF, true_residual=True)
    assert res["rel_resid"] <= 1e-10
