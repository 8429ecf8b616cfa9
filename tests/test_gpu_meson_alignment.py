"""GPU: propagators of cmx_meson_2pt_noalloc that start on 8 but not on 16 bytes, which the kernel's 16-byte direct
loads to LDS must not be given, against the same propagators on 16 bytes, bit for bit."""
import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.test_zz_no_alloc import Hip, noalloc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,nmom", [((4, 4, 6, 6), 1), ((6, 2, 10, 4), 5)])
def test_meson_alignment(L, nmom):
    V = int(np.prod(L))
    r = np.random.default_rng(8)
    S = [r.standard_normal((V, 12, 12)) + 1j * r.standard_normal((V, 12, 12)) for _ in range(2)]
    moms = r.integers(-2, 3, (nmom, 3)).astype(np.int32)
    hip = Hip()
    try:
        on16 = [hip.upload(s) for s in S]
        on8 = [hip.upload(np.concatenate([[0.0], s.view(np.float64).ravel()])) for s in S]
        on8 = [type(p)(p.value + 8) for p in on8]
        dm = hip.upload(moms)
        for k in (0, 1):  # one propagator, and two
            want = cmx.meson_2pt(L, S[0], S[1] if k else None, (1, 0, 1, 2), moms)
            for a, b in ((on16[0], on16[k]), (on8[0], on8[k]), (on16[0], on8[k]), (on8[0], on16[k])):
                print("meson alignment", L, nmom, a.value % 16, b.value % 16, flush=True)
                dout = hip.empty(want.nbytes)
                cmx.check(noalloc(hip, L, a, b, (1, 0, 1, 2), dm, nmom, dout))
                assert hip.download(dout, np.zeros_like(want)).tobytes() == want.tobytes()
    finally:
        hip.free()
