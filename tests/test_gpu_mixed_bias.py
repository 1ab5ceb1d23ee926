"""Mixed-precision builds: the FP32 quartets' rounding errors must not add up.
Rounding to nearest has no preferred sign, so the energy error 1/2 tr D dG of a
build with N independent errors grows like their root mean square, not like their
sum.  With e = w D dG per packed element (w = 2 off the diagonal), |sum e| stays
below 3 sqrt(2) sqrt(sum e^2): three standard deviations, and sqrt(2) because the
error of one integral (ij|kl) reaches tr D dG through two elements with the same
weight (J_ij and J_kl, K_ik and K_jl).  FP32 sums that run from the largest
primitive to the smallest lose the small ones with their sign and fail this (7 to
10 times the root mean square)."""
import numpy as np
import pytest

from openqp_amd import basis as B, molecules as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [1, 2])
def test_mixed_energy_error_is_unbiased(seed):
    from openqp_amd import lib as L
    print("mixed bias (H2O)32/cc-pVDZ seed", seed, flush=True)
    Z, xyz = M.water_grid(4, 4, 2, seed=seed)
    bas = B.build_basis("cc-pvdz", Z, xyz)
    S, _, _ = L.int1e(bas)
    dp = B.pack_tri(M.random_density(S, 160, seed=seed + 10))
    fb = L.FockBuilder(bas)
    ref = fb.fock_jk(dp)
    fb.set_precision(1, 1e-3)
    mixed = fb.fock_jk(dp)
    assert fb.last_stats.quartets_fp32 > 0
    fb.close()
    w = np.full(dp.size, 2.0)
    i = np.arange(bas.nbf)
    w[i * (i + 1) // 2 + i] = 1.0
    e = w * dp * (mixed - ref)
    z = abs(e.sum()) / np.sqrt((e * e).sum())
    print("  dE2", 0.5 * e.sum(), "against the root mean square:", z, flush=True)
    assert z <= 3.0 * np.sqrt(2.0)
