"""GPU: the clover force's work-groups (64 sites of a checkerboard, the four directions of each) on lattices that
fill them partly and on extents of 2, where a site's neighbour on both sides is the same, against the oracle."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.util import random_fermion, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(2, 2, 2, 2), (2, 4, 6, 2), (4, 6, 2, 10), (6, 2, 10, 14)])
def test_force_edges(L):
    print("force edges", L, flush=True)
    V = int(np.prod(L))
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=7, eps=0.4), (1, 1, 1, -1))
    mass = cmx.kappa_to_mass(0.12)
    op = cmx.Operator(cmx.Gauge(L, U), cmx.EO_CLOVER, mass, 1.0, 1.2)
    chi, psi = random_fermion(V, 1), random_fermion(V, 2)
    # a link's derivative adds 24 terms of products of 12 factors of size one and spin sums of 4: rounding of a
    # few hundred eps at most
    for cb in (0, 1):
        assert rel(op.clover_deriv(chi, psi, cmx.PLUS, cb), oracle.clover_deriv(L, U, chi, psi, 1.0, 1.2, cb)) < 1e-13
    assert rel(op.clover_deriv_trln(), oracle.clover_deriv_trln(L, U, mass, 1.0, 1.2)) < 1e-13
    lo = slice(V // 2, None)
    got = op.deriv(chi[lo], psi[lo], cmx.PLUS)
    c, p = chi.copy(), psi.copy()
    c[: V // 2] = 0
    p[: V // 2] = 0
    assert rel(got, oracle.eo_clover_deriv(L, U, mass, c, p, +1, 1.0, 1.2)) < 1e-13
