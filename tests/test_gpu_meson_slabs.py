"""GPU: propagators of more than 1 GiB, which cmx_meson_2pt takes through the device in ranges of time slices (here 14 and
2 of 16), against the same propagators whole on the device, bit for bit."""
import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.test_zz_no_alloc import Hip, noalloc

pytestmark = pytest.mark.gpu


def test_meson_slabs():
    L, origin = (32, 32, 32, 16), (1, 2, 3, 4)
    V = int(np.prod(L))
    r = np.random.default_rng(8)
    S = [(r.random((V, 144, 2)) - 0.5).view(np.complex128).reshape(V, 12, 12) for _ in range(2)]
    moms = np.array([(0, 0, 0), (1, 0, 0), (0, -1, 1)], np.int32)
    hip = Hip()
    try:
        d = [hip.upload(s) for s in S]
        dm = hip.upload(moms)
        for k in (0, 1):  # one propagator, and two
            print("meson slabs", L, k, flush=True)
            got = cmx.meson_2pt(L, S[0], S[1] if k else None, origin, moms)
            dout = hip.empty(got.nbytes)
            cmx.check(noalloc(hip, L, d[0], d[k], origin, dm, len(moms), dout))
            assert hip.download(dout, np.zeros_like(got)).tobytes() == got.tobytes()
    finally:
        hip.free()
