"""GPU: the one-pass meson contraction at the sizes where its ranges end: slices that are no multiple of 16
sites, work-group ranges that cross the checkerboards, 1 to 70 momenta (passes of 1, 2, 4 and 8, and a second
pass of momenta), negative and large momentum numbers, odd origins; against the oracle.  Both sides sum in
FP64: 2e3 to 3e4 terms per number leave rel below 1e-13."""
import numpy as np
import pytest

import oracle
from chroma_amd import lib as cmx
from tests.util import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,nmom,same", [((2, 2, 2, 2), 1, True), ((2, 6, 2, 4), 2, False), ((6, 6, 10, 4), 3, True),
                                         ((10, 6, 6, 2), 5, False), ((14, 10, 6, 2), 9, True), ((4, 4, 6, 6), 70, False)])
def test_meson_ranges(L, nmom, same):
    V = int(np.prod(L))
    r = np.random.default_rng(17)
    S1 = r.standard_normal((V, 12, 12)) + 1j * r.standard_normal((V, 12, 12))
    S2 = None if same else r.standard_normal((V, 12, 12)) + 1j * r.standard_normal((V, 12, 12))
    moms = r.integers(-20, 21, (nmom, 3))
    origin = tuple(int(v) for v in (np.array(L) * 3 // 4))
    print("meson ranges", L, nmom, same, origin, flush=True)
    got = cmx.meson_2pt(L, S1, S2, origin, moms)
    assert rel(got, oracle.mesons(L, S1, S2, origin, moms)) < 1e-13
