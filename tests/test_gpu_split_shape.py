"""GPU: the direction-split kernel by name.  A shape that was read can be set again without changing the kernel or a
bit of the result; the kernel asked for is the one reported; and it agrees with the oracle on both sides of the size
up to which FP16 operators choose it by themselves, with a last work-group that is partly empty."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.test_gpu_parity import TOL
from tests.util import random_fermion, rel

pytestmark = pytest.mark.gpu

SPLIT = 5


def make_op(L, kind=cmx.EO_CLOVER, sloppy=cmx.HALF, **kw):
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=5, eps=0.3), (1, 1, 1, -1))
    return U, cmx.Operator(cmx.Gauge(L, U), kind, cmx.kappa_to_mass(0.11), 1.0, sloppy_prec=sloppy, **kw)


def test_read_shape_can_be_set():
    L = (4, 6, 4, 10)
    Vh = int(np.prod(L)) // 2
    _, op = make_op(L)
    psi = random_fermion(2 * Vh, 3)[Vh:]
    for prec in (cmx.DOUBLE, cmx.SINGLE, cmx.HALF):
        before = op(psi, +1, prec).tobytes(), op.dslash(psi, +1, 0, prec).tobytes()
        shapes = [op.hop_config(prec, t) for t in (1, 2)]
        assert shapes[0]["fast"] == SPLIT and shapes[1]["fast"] == (1 if prec == cmx.HALF else SPLIT)
        for t in (1, 2):
            op.set_hop_config(prec, target=t, **shapes[t - 1])
        assert [op.hop_config(prec, t) for t in (1, 2)] == shapes
        assert before == (op(psi, +1, prec).tobytes(), op.dslash(psi, +1, 0, prec).tobytes())
    for fast in (4, 6, 7, 8, -1):
        with pytest.raises(cmx.CmxError):
            op.set_hop_config(cmx.SINGLE, 64, 0, 1, 0, fast)


def test_not_admitted():
    L = (4, 4, 4, 8)
    _, op = make_op(L, sloppy=cmx.SINGLE, sloppy_recon=cmx.RECONS_18)
    op.set_hop_config(cmx.SINGLE, 64, 0, 1, 0, SPLIT)
    assert op.hop_config(cmx.SINGLE)["fast"] == 0


@pytest.mark.parametrize("L", [(4, 6, 2, 10), (16, 16, 16, 18), (12, 10, 14, 50)])
@pytest.mark.parametrize("kind", [cmx.UNPREC_WILSON, cmx.EO_CLOVER])
def test_split_against_oracle(L, kind):
    V = int(np.prod(L))
    psi = random_fermion(V, 6)
    lo = 0 if kind == cmx.UNPREC_WILSON else V // 2
    U, op = make_op(L, kind)
    ref_op = oracle.Op(kind, L, U, cmx.kappa_to_mass(0.11), 1.0, 1.0)
    ref = [ref_op(psi, isign)[lo:] for isign in (+1, -1)]
    for prec in (cmx.DOUBLE, cmx.SINGLE, cmx.HALF):
        op.set_hop_config(prec, 64, 0, 1, 0, SPLIT, target=1)
        print("split", L, kind, prec, flush=True)
        assert op.hop_config(prec)["fast"] == SPLIT
        for k, isign in enumerate((+1, -1)):
            assert rel(op(psi[lo:], isign, prec), ref[k]) < TOL[prec]
