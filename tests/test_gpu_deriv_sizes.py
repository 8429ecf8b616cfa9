"""GPU: the hopping term's link derivative on both sides of the size from which each direction's part is copied to its
place by itself (1820 sites per checkerboard), against the oracle."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.util import random_fermion, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(2, 2, 2, 2), (4, 4, 8, 24), (8, 8, 8, 8)])
def test_deriv_sizes(L):
    V = int(np.prod(L))
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=3, eps=0.3), (1, 1, 1, -1))
    op = cmx.Operator(cmx.Gauge(L, U), cmx.EO_WILSON, 0.1)
    chi, psi = random_fermion(V, 1), random_fermion(V, 2)
    for cb in (0, 1, -1):
        print("deriv sizes", L, cb, flush=True)
        # a sum of eight products per number
        assert rel(op.dslash_deriv(chi, psi, +1, cb), oracle.dslash_deriv(L, chi, psi, +1, cb)) < 1e-14
