"""The cooperative gradient kernel (k_gradc) and the split form of the per-lane
templates (several lanes per ket) against the oracle (1e-8, the bound of the
gradient tests) and, with the kernel off (OQPH_GRADC=0), the same quartet and
primitive counts and forces to 1e-11 (sums of up to 1e5 terms below 1e1 in
another order: 1e5 * 1e1 * 1e-16 = 1e-10 at worst, its square root in practice).
One water fills few lane groups and splits every ket; s and p only, Cartesian
and pure d, f; a density with both shells of a pair on one atom."""
import numpy as np
import pytest

from helpers import density_for, small_system
from openqp_amd import basis as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,nw,harmonic", [("6-31g", 1, None), ("6-31g", 4, None), ("6-31g(d)", 1, None),
                                               ("6-31g(d)", 3, None), ("cc-pvdz", 2, 0), ("cc-pvtz", 1, None),
                                               ("cc-pvtz", 1, 0), ("cc-pvtz", 2, None)])
def test_cooperative_and_split_gradient(oracle, monkeypatch, basis, nw, harmonic):
    from openqp_amd import lib as L
    print("k_gradc", basis, nw, harmonic, flush=True)
    bas = small_system(basis, nw=nw, seed=5)
    if harmonic is not None:
        bas = B.build_basis(basis, bas.zn.astype(int), bas.xyz, harmonic=harmonic)
    _, dp = density_for(oracle, bas, 5 * nw, seed=8)
    go, _ = oracle.grad2(bas, dp)
    out = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("OQPH_GRADC", mode)
        fb = L.FockBuilder(bas)
        g = np.asarray(fb.grad2(dp))
        st = fb.last_stats
        out[mode] = (g, st.quartets_computed, st.quartets_screened, st.prim_quartets)
        print("  OQPH_GRADC", mode, "max |g - g_oracle| =", np.abs(g - go).max(), out[mode][1:], flush=True)
        assert np.abs(g - go).max() <= 1e-8
        fb.close()
    assert out["0"][1:] == out["1"][1:]
    assert np.abs(out["0"][0] - out["1"][0]).max() <= 1e-11
