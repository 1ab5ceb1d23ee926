"""Device memory of prepared sessions with long primitive lists and no s shells:
the primitive-pair records (48 bytes in FP64, 24 in FP32) and little else.  The
piecewise copies that kets of two s shells are read from (72 bytes more per record)
are not made for pairs that no kernel reads that way.  The bases are p shells of 12
primitives with every primitive pair above the cutoffs, so n of them have n (n + 1) / 2
pairs of 144 records.  From 60 to 240 shells a session may grow by the records, by 512
bytes a pair (its record of about 130 bytes, the AO block of 72 in four buffers, index
lists) and by 64 MiB (the device allocates whole pages of 2 MiB, for 32 buffers); the
copies alone would be 3.5 times that allowance."""
import ctypes as C

import numpy as np
import pytest

from helpers import DeviceBuffer
from openqp_amd import basis as B

pytestmark = pytest.mark.gpu


def _free():
    free, total = C.c_size_t(), C.c_size_t()
    hip = DeviceBuffer.hip()
    hip.hipDeviceSynchronize()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _basis(nsh, nprim):
    i32 = lambda v: np.asarray(v, np.int32)
    ex = np.tile(np.geomspace(0.2, 2.0, nprim), nsh)
    cc = np.full(nsh * nprim, 0.1)
    xyz = np.random.default_rng(5).uniform(-1.0, 1.0, (nsh // 2, 3))
    return B.Basis("p only", i32([1] * nsh), i32([0] * nsh), i32([s // 2 for s in range(nsh)]), i32([nprim] * nsh),
                   i32(range(0, nsh * nprim, nprim)), i32(range(0, 3 * nsh, 3)), ex, cc, xyz, np.ones(nsh // 2))


def test_prepared_session_holds_little_beside_the_records():
    from openqp_amd import lib as L
    nprim = 12
    pairs = lambda n: n * (n + 1) // 2
    used = {}
    builders = [L.FockBuilder(_basis(4, 2))]  # code objects and tables are loaded before the first reading
    builders[0].prepare()
    for nsh in (60, 240):
        print("session memory", nsh, "p shells of", nprim, flush=True)
        bas = _basis(nsh, nprim)
        before = _free()
        builders.append(L.FockBuilder(bas))
        builders[-1].prepare()
        used[nsh] = before - _free()
    for fb in builders:
        fb.close()
    np_ = pairs(240) - pairs(60)
    records = 72 * np_ * nprim * nprim
    print("  records", records, "bytes, sessions", used, flush=True)
    assert used[240] - used[60] >= records - (64 << 20)
    assert used[240] - used[60] <= records + 512 * np_ + (64 << 20)
