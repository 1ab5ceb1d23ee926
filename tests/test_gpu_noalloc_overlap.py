"""A no-allocation build keeps all of its device memory in an array of its own, so it
may run while a device build of the same session is still in flight on another
stream: both are issued without statistics (nothing then waits for the device),
with densities of different size, and each result is that of the build alone.  Two
runs of one build differ by the order of FP64 atomic sums only: 1e-12, the bound of
the other no-allocation tests, per unit of the largest density element."""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceBuffer, density_for, small_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,nw", [("6-31g", 2), ("cc-pvdz", 4)])
def test_noalloc_beside_a_device_build(oracle, basis, nw):
    from openqp_amd import lib as L
    print("no-alloc beside a device build", basis, nw, flush=True)
    bas = small_system(basis, nw=nw, seed=7)
    fb = L.FockBuilder(bas)
    fb.prepare()
    _, d1 = density_for(oracle, bas, 5 * nw, seed=11)
    _, d2 = density_for(oracle, bas, 5 * nw, seed=12)
    d2 = 64.0 * d2
    hip = DeviceBuffer.hip()
    streams = [C.c_void_p(), C.c_void_p()]
    for s in streams:
        assert hip.hipStreamCreate(C.byref(s)) == 0
    bufs = [DeviceBuffer(d1.size) for _ in range(4)]
    a, b, fa, fn = bufs
    a.upload(d1)
    b.upload(d2)
    fb.fock_jk_device(a.address, fa.address)
    fb.fock_jk_device(b.address, fn.address)
    ref1, ref2 = fa.download(), fn.download()
    lib = L.load()
    for i in range(6):
        fa.upload(np.zeros(d1.size))
        fn.upload(np.zeros(d1.size))
        assert lib.oqph_fock_jk_device(fb._s, C.c_void_p(a.address), C.c_void_p(fa.address), 1, 1.0, 1.0, None,
                                       streams[0]) == 0
        assert lib.oqph_fock_jk_noalloc(fb._s, C.c_void_p(b.address), C.c_void_p(fn.address), 1.0, 1.0, None,
                                        streams[1]) == 0
        hip.hipDeviceSynchronize()
        e1, e2 = np.abs(fa.download() - ref1).max(), np.abs(fn.download() - ref2).max()
        print("  pass", i, "device build", e1, "no-alloc build", e2, flush=True)
        assert e1 <= 1e-12 * max(1.0, np.abs(d1).max())
        assert e2 <= 1e-12 * max(1.0, np.abs(d2).max())
    for s in streams:
        hip.hipStreamDestroy(s)
    for x in bufs:
        x.free()
    fb.close()
