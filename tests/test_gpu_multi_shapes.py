"""GPU: the multi-source hop equals the single-source hop bit for bit with the launch shapes that an operator has of
itself, untuned and autotuned, on lattices small enough for its other kernels to be direction-split."""
import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.util import random_fermion

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(8, 8, 8, 16), (16, 16, 8, 16), (6, 4, 8, 10)])
@pytest.mark.parametrize("autotune", [False, True])
def test_dslash_multi_own_shapes(L, autotune):
    print("dslash multi own shapes", L, autotune, flush=True)
    Vh = int(np.prod(L)) // 2
    U = cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=21, eps=0.3), (1, 1, 1, -1))
    op = cmx.Operator(cmx.Gauge(L, U), cmx.EO_WILSON, 0.1, sloppy_prec=cmx.HALF, autotune=autotune)
    src = np.stack([random_fermion(2 * Vh, 300 + k)[:Vh] for k in range(5)])
    for group in (0, 1, 4):
        op.set_multi_group(group)
        for cb in (0, 1):
            for isign in (+1, -1):
                got = op.dslash_multi(src, isign, cb, cmx.HALF)
                for k in range(5):
                    assert got[k].tobytes() == op.dslash(src[k], isign, cb, cmx.HALF).tobytes(), (group, cb, isign, k)
