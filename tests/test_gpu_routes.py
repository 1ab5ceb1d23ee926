"""Which kernels a gradient and a response pass ran: the cooperative and split gradient
kernels and the dense response pass where their rules send a class or a size, and the
ones they replace when they are switched off, so that the tests that compare the two
sides do compare two kernels."""
import numpy as np
import pytest

from helpers import density_for, small_system
from openqp_amd.basis import ncart
from openqp_amd.build import GRC

pytestmark = pytest.mark.gpu
COOP = {1000 * a + 100 * b + 10 * c + d for a, b, c, d in GRC}


def _components(c):
    return ncart(c // 1000) * ncart(c // 100 % 10) * ncart(c // 10 % 10) * ncart(c % 10)


@pytest.mark.parametrize("basis,nw", [("6-31g", 1), ("6-31g(d)", 1), ("6-31g(d)", 3), ("cc-pvtz", 1)])
def test_gradient_kernels(oracle, monkeypatch, basis, nw):
    from openqp_amd import lib as L
    print("gradient kernels", basis, nw, flush=True)
    bas = small_system(basis, nw=nw, seed=5)
    _, dp = density_for(oracle, bas, 5 * nw, seed=8)
    for mode in ("0", "1"):
        monkeypatch.setenv("OQPH_GRADC", mode)
        fb = L.FockBuilder(bas)
        assert fb.last_gradient_kernels() == []
        fb.grad2(dp)
        ran = fb.last_gradient_kernels()
        fb.close()
        print("  OQPH_GRADC", mode, sorted(ran), flush=True)
        kern = dict(ran)
        large = [c for c, k in ran if k == "k_gradc"]
        if mode == "0":
            assert not large
        else:
            # every class that has a cooperative kernel, all above 64 components
            assert large and min(_components(c) for c in large) > 64
            assert set(large) == {c for c, _ in ran if c in COOP}
        # a few wavefronts of contracted s quartets: several lanes per ket
        assert kern[0] == "k_grad_split"


@pytest.mark.parametrize("mode,nf", [("0", 1), ("1", 1), ("1", 5)])
def test_response_route(monkeypatch, mode, nf):
    from openqp_amd import lib as L
    print("response route", mode, nf, flush=True)
    monkeypatch.setenv("OQPH_RESPONSE", mode)
    bas = small_system("6-31g", nw=2, seed=5)
    fb = L.FockBuilder(bas)
    assert fb.last_response_dense() is None
    fb.mrsf_int2(0.1 * np.random.default_rng(2).standard_normal((bas.nbf, bas.nbf, 7, nf)))
    assert fb.last_response_dense() is (mode == "1")
    fb.close()
