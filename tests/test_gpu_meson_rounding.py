"""GPU: the rounding of coherent meson sums.  The pion of one propagator at zero momentum is sum |S|^2, all terms
positive, so the error of every partial sum is visible; against extended precision on the host."""
import numpy as np
import pytest

from chroma_amd import lib as cmx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(8, 10, 6, 8), (12, 12, 12, 2)])
def test_pion_rounding(L):
    V = int(np.prod(L))
    r = np.random.default_rng(3)
    S = r.standard_normal((V, 12, 12)) + 1j * r.standard_normal((V, 12, 12))
    print("pion rounding", L, flush=True)
    got = cmx.meson_2pt(L, S, None, (0, 0, 0, 0), [[0, 0, 0]])[15, 0].real
    site = (S.real.astype(np.longdouble) ** 2 + S.imag.astype(np.longdouble) ** 2).reshape(V, -1).sum(1)
    want = site.reshape(2, L[3], -1).sum(axis=(0, 2))  # checkerboard-major, t slowest within a checkerboard
    # In units of 2^-53: a work-group's sum is off by about one (16 spins in one chain: 0.6 sqrt(16 / 3) rms, averaged
    # over its lanes), the compensated sum over 30 and 108 work-groups averages that to below 0.3, and the last rounding
    # adds one at most.  3 leaves six times the rms; summing the work-groups plainly adds 0.6 sqrt(30 / 3) rms or more.
    assert np.max(np.abs(got - want) / want) < 3 * 2.0 ** -53
