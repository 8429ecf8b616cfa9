"""GPU: the device-resident multishift recurrences at one shift, at the most shifts, with shifts that stop early,
and at MaxIter."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.util import random_fermion, rel

pytestmark = pytest.mark.gpu

L = (4, 6, 2, 8)


def setup():
    V = int(np.prod(L))
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=5, eps=0.3), (1, 1, 1, -1))
    mass = cmx.kappa_to_mass(0.12)
    chi = random_fermion(V, 8)
    chi[: V // 2] = 0
    return cmx.Operator(cmx.Gauge(L, U), cmx.EO_CLOVER, mass, 1.0), oracle.Op(oracle.EO_CLOVER, L, U, mass, 1.0, 1.0), chi


@pytest.mark.parametrize("shifts", [[0.01], list(np.geomspace(1e-3, 1e3, 64)), [50.0, 0.1, 1e4, 0.1]])
def test_shift_counts(shifts):
    print("multishift", len(shifts), flush=True)
    op, ref, chi = setup()
    psi, res = op.solve_multishift(chi[chi.shape[0] // 2:], shifts, rsd=1e-10, maxit=200)
    want, n, _ = ref.solve_multishift(chi, shifts, 1e-10, maxit=200)
    assert abs(res[0]["n_count"] - n) <= 1  # rounding in the last test
    for k in range(len(shifts)):
        # both stop at |r_s| <= 1e-10 |chi|: they differ by at most twice that times the condition number
        # of M^dag M, below 900
        assert rel(psi[k], want[k][chi.shape[0] // 2:]) < 2 * 900 * 1e-10


@pytest.mark.parametrize("rsd", [1e-1, 1e-3, 1e-5, 1e-7, 1e-9])
def test_maxit(rsd):
    """Solves of different lengths, so that the last iteration falls on different places between two host reads:
    the length has to stay below MaxIter (minvcg2.cc:357-359), and the operator solves normally after an error."""
    op, _, chi = setup()
    chi = chi[chi.shape[0] // 2:]
    want, res = op.solve_multishift(chi, [0.01, 1.0], rsd=rsd, maxit=200)
    n = res[0]["n_count"]
    print("multishift maxit", rsd, n, flush=True)
    for maxit in (n, max(1, n - 1)):
        with pytest.raises(cmx.CmxError):
            op.solve_multishift(chi, [0.01, 1.0], rsd=rsd, maxit=maxit)
    got, res = op.solve_multishift(chi, [0.01, 1.0], rsd=rsd, maxit=n + 1)
    assert res[0]["n_count"] == n and got.tobytes() == want.tobytes()
