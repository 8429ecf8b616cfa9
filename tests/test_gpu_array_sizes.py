"""GPU: host arrays whose size is not the operator's subset.  Longer ones give the result of the leading part and
zeros behind it (stout smearing: the links behind it); shorter ones, which the library would read or write past the
end, are refused."""
import numpy as np
import pytest

from chroma_amd import lib as cmx
from tests.util import random_fermion

pytestmark = pytest.mark.gpu

L = (4, 4, 2, 6)
V = int(np.prod(L))


@pytest.fixture(scope="module")
def links():
    return cmx.gauge_apply_bc(L, cmx.gauge_generate(L, kind=1, seed=5, eps=0.3), (1, 1, 1, -1))


@pytest.fixture(scope="module")
def op(links):
    return cmx.Operator(cmx.Gauge(L, links), cmx.EO_WILSON, cmx.kappa_to_mass(0.11), sloppy_prec=cmx.HALF)


def calls(op):
    net = cmx.Net()
    net.init_neumann(4.1)
    cmx.net_attach(op, net)
    return {"apply": lambda a: op(a), "dslash": lambda a: op.dslash(a, +1, 0),
            "multi": lambda a: op.dslash_multi(a[None], +1, 0)[0], "solve": lambda a: op.solve(a, rsd=1e-6)[0],
            "guess": lambda a: op.solve(a, psi=0 * a, rsd=1e-6)[0],
            "multishift": lambda a: op.solve_multishift(a, [0.1], rsd=1e-6)[0][0],
            "batch": lambda a: cmx.solve_batch([op], [a], rsd=1e-4, tune=False)[0][0],
            "net": lambda a: cmx.net_apply(op, a)}


def test_sizes(op):
    chi = random_fermion(V, 3)[V // 2:]
    for name, f in calls(op).items():
        print("sizes", name, flush=True)
        want = f(chi)
        for _ in range(3):  # a fresh allocation may hold zeros by chance
            junk = np.full((V, 4, 3), 7.0 + 3.0j)
            del junk
            got = f(np.concatenate([chi, chi]))
            assert got.shape == (V, 4, 3) and got[: V // 2].tobytes() == want.tobytes(), name
            assert not got[V // 2:].any(), name
        with pytest.raises(ValueError):
            f(chi[:-1])


def test_links(links):
    want = cmx.gauge_stout_smear(L, links, 1, 0.1)
    long = np.concatenate([links, links[:1] + 1])
    got = cmx.gauge_stout_smear(L, long, 1, 0.1)
    assert got.shape == long.shape and got[:4].tobytes() == want.tobytes() and (got[4:] == long[4:]).all()
    with pytest.raises(ValueError):
        cmx.gauge_stout_smear(L, links[:3], 1, 0.1)
