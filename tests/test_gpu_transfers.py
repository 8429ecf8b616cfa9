"""GPU: host arrays on both sides of the sizes where the staging changes (one to four threads, one or several
pinned slots), with runs of zeros that are cleared on the device instead of sent, bit for bit; and the entry
points that start from zero against an explicit zero guess."""
import threading

import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.util import random_fermion

pytestmark = pytest.mark.gpu

# checkerboards of 0.05, 0.07, 0.98, 1.08, 3.98, 4.4, 7.96, 8.8 and 16.7 MB
LATTICES = [(4, 4, 4, 8), (4, 4, 6, 8), (8, 8, 8, 20), (8, 8, 8, 22), (12, 12, 16, 18), (12, 12, 16, 20), (16, 16, 18, 18), (16, 16, 18, 20),
            (16, 16, 20, 34)]


def make_op(L, kind=cmx.EO_WILSON):
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=2, eps=0.3), (1, 1, 1, -1))
    return cmx.Operator(cmx.Gauge(L, U), kind, cmx.kappa_to_mass(0.11))


@pytest.mark.parametrize("L", LATTICES)
def test_roundtrip_bits(L):
    print("transfer", L, flush=True)
    n = int(np.prod(L)) // 2
    op = make_op(L)
    rng = np.random.default_rng(1)
    x = rng.normal(size=(n, 4, 3)) + 1j * rng.normal(size=(n, 4, 3))
    sparse = x.copy()
    sparse[n // 8:] = 0
    sparse[-1, 3, 2] = complex(0.0, -0.0)  # not zero bits: must arrive
    point = np.zeros_like(x)
    point[n // 2, 1, 1] = 1
    for a in (x, sparse, point, np.zeros_like(x)):
        assert op.layout_roundtrip(a, cmx.DOUBLE).tobytes() == a.tobytes()


def test_roundtrip_threads():
    L = (12, 12, 16, 20)
    n = int(np.prod(L)) // 2
    got = {}

    def work(k):
        op = make_op(L)
        a = np.random.default_rng(k).normal(size=(n, 4, 3)) + 0j
        got[k] = all(op.layout_roundtrip(a, cmx.DOUBLE).tobytes() == a.tobytes() for _ in range(3))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert got == {k: True for k in range(6)}


@pytest.mark.parametrize("solver,sloppy", [(cmx.CG, cmx.DOUBLE), (cmx.RELIABLE_CG, cmx.HALF),
                                           (cmx.RELIABLE_BICGSTAB, cmx.SINGLE), (cmx.FGMRESDR, cmx.SINGLE)])
def test_from_zero(solver, sloppy):
    L = (4, 6, 4, 8)
    print("from zero", solver, sloppy, flush=True)
    op = make_op(L)
    chi = random_fermion(int(np.prod(L)), 4)[int(np.prod(L)) // 2:]
    a, ra = op.solve(chi, solver=solver, rsd=1e-9, sloppy_prec=sloppy)
    b, rb = op.solve(chi, psi=np.zeros_like(chi), solver=solver, rsd=1e-9, sloppy_prec=sloppy)
    assert a.tobytes() == b.tobytes() and ra["n_count"] == rb["n_count"]


def test_batch_from_zero_and_repeated_shape():
    """The second tuned batch of the same make-up takes the shape of the first."""
    L = (4, 6, 4, 8)
    op = make_op(L)
    chis = [random_fermion(int(np.prod(L)), 10 + k)[int(np.prod(L)) // 2:] for k in range(3)]
    runs = [cmx.solve_batch([op] * 3, chis, psis=z, rsd=1e-9, sloppy_prec=cmx.HALF)
            for z in (None, [np.zeros_like(c) for c in chis], None)]
    for psis, res, summary in runs[1:]:
        assert [p.tobytes() for p in psis] == [p.tobytes() for p in runs[0][0]]
        assert (summary["hop_block"], summary["hop_fast"]) == (runs[0][2]["hop_block"], runs[0][2]["hop_fast"])
