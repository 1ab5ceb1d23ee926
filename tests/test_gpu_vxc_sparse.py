"""Vxc of two waters far apart: V is block diagonal with the blocks of the single waters,
E_xc and the electron count are their sums.  The grid's boxes span the gap (8e9 of them
for (4000, 4000, 4000) bohr; 5e19, beyond a 64-bit index, for 7.5e6 bohr), so a table
with an entry per box must not be needed.  Bound: coordinates of size X carry a rounding
of X eps / 2, which moves a function of slope up to 1e3 by 1e3 X eps on a few thousand
points of weighted density below 1: 1e3 4000 2.2e-16 1e3 = 1e-6 at worst and 1e-8 with
random signs for the first, times 2000 for the second, where only the electron count is
compared, to 1e-4."""
import numpy as np
import pytest

from helpers import small_system
from openqp_amd import basis as B, molecules as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [4.0e3, 7.5e6])
def test_far_fragments(oracle, shift):
    from openqp_amd.lib import FockBuilder
    print("vxc of far fragments", shift, flush=True)
    one = small_system("6-31g(d)", nw=1)
    S, _, _ = oracle.int1e(one)
    D = M.random_density(S, 5, seed=7)
    fb = FockBuilder(one)
    fb.set_xc("b3lyp5", 20, 6)
    V1, e1, n1 = fb.vxc(B.pack_tri(D))
    fb.close()
    V1 = B.unpack_tri(V1[0], one.nbf)
    two = B.build_basis("6-31g(d)", np.concatenate([one.zn, one.zn]).astype(int),
                        np.concatenate([one.xyz, one.xyz + shift]))
    n = one.nbf
    D2 = np.zeros((2 * n, 2 * n))
    D2[:n, :n] = D2[n:, n:] = D
    fb = FockBuilder(two)
    fb.set_xc("b3lyp5", 20, 6)
    V2, e2, n2 = fb.vxc(B.pack_tri(D2))
    fb.close()
    V2 = B.unpack_tri(V2[0], 2 * n)
    err = max(np.abs(V2[:n, :n] - V1).max(), np.abs(V2[n:, n:] - V1).max())
    print("  max |dV|", err, "dE", e2 - 2 * e1, "dN", n2 - 2 * n1, flush=True)
    assert np.abs(V2[:n, n:]).max() == 0.0
    assert np.isfinite(V2).all() and abs(n2 - 2 * n1) < 1e-4
    if shift < 1e5:
        assert err < 1e-8 and abs(e2 - 2 * e1) < 1e-8 and abs(n2 - 2 * n1) < 1e-8
