"""GPU: the stout step's work-groups (64 sites of a checkerboard, all four directions) on lattices that fill
them partly, and exp(iQ) from the norm 0 to norms that need several squarings, against the oracle."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.util import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,rho,dirs", [((2, 2, 2, 2), 0.1, 15), ((2, 4, 6, 2), 0.3, 11), ((4, 6, 2, 10), 0.8, 15),
                                        ((6, 2, 10, 14), 4.0, 13), ((4, 4, 4, 2), 0.1, 0), ((4, 4, 4, 2), 1e-9, 15)])
def test_stout_edges(L, rho, dirs):
    print("stout edges", L, rho, dirs, flush=True)
    U = cmx.gauge_generate(L, kind=2, seed=3)
    got = cmx.gauge_stout_smear(L, U, 1, rho, dirs)
    # |Q|_F <= 6 sqrt(3) rho; s squarings of unit-size matrices double the rounding (a few eps) each time
    tol = 1e-14 * max(1.0, 6 * np.sqrt(3) * rho)
    assert rel(got, oracle.stout(L, U, rho, 1, dirs)) < tol
