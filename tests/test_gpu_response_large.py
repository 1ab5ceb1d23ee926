"""Response passes of many densities.  The caller's array passes through the density and
output slabs of the pass: a pass may hold 2 slabs of nd nbf^2 doubles more than one of
few densities, and 16 MiB (whole pages of 2 MiB, the density flags).  More elements than
one sweep of the packing kernels (16384 blocks of 256): each density's result is that of
a pass with fewer of them, to 1e-12 (the same integrals and products, elements below 10,
summed in another order); the last component, which the screens read, is the same for
all."""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceBuffer, small_system

pytestmark = pytest.mark.gpu


def _free():
    free, total = C.c_size_t(), C.c_size_t()
    hip = DeviceBuffer.hip()
    hip.hipDeviceSynchronize()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("mode", ["0", "1"])
def test_many_densities(monkeypatch, mode):
    from openqp_amd import lib as L
    monkeypatch.setenv("OQPH_RESPONSE", mode)
    bas = small_system("6-31g", nw=8, seed=5)
    n, nmat, nf = bas.nbf, 7, 60
    print("response pass of many densities, OQPH_RESPONSE", mode, "nbf", n, flush=True)
    assert n * n * nmat * nf > 16384 * 256
    rng = np.random.default_rng(3)
    d3 = 0.1 * rng.standard_normal((n, n, nmat, nf))
    d3[:, :, -1, :] = d3[:, :, -1, :1]
    fb = L.FockBuilder(bas)
    few = fb.mrsf_int2(np.ascontiguousarray(d3[:, :, :, :3]))
    before = _free()
    many = fb.mrsf_int2(d3)
    grown = before - _free()
    fb.close()
    slab = 8 * n * n * nmat * nf
    print("  slab", slab, "grown by", grown, "max |difference|", np.abs(many[:, :, :, :3] - few).max(), flush=True)
    assert grown <= 2 * slab * (((n + 15) & ~15) / n) + (16 << 20)
    assert np.abs(many[:, :, :, :3] - few).max() <= 1e-12
    assert np.abs(many[:, :, -1, :] - many[:, :, -1, :1]).max() <= 1e-12
