"""A launch of the cooperative J/K kernel with more than 65536 blocks (several rows of
its grid) against the kernels it replaces (OQPH_JKC=0): equal quartet counts, and G to
1e-11 (different order of at most 1e7 FP64 terms below 1 per element: 1e7 eps = 2e-9 at
worst, its square root in practice)."""
import numpy as np
import pytest

from openqp_amd import basis as B, molecules as M

pytestmark = pytest.mark.gpu


def test_many_blocks(monkeypatch):
    from openqp_amd import lib as L
    print("k_jkc with several grid rows, (H2O)8/cc-pVTZ", flush=True)
    Z, xyz = M.water_grid(2, 2, 2, seed=3)
    bas = B.build_basis("cc-pvtz", Z, xyz)
    S, _, _ = L.int1e(bas)
    dp = B.pack_tri(M.random_density(S, 40, seed=4))
    out = {}
    for mode in ("0", "2"):
        monkeypatch.setenv("OQPH_JKC", mode)
        fb = L.FockBuilder(bas)
        fb.set_profiling(True)
        f = fb.fock_jk(dp)
        waves = max([p["slots"] // 64 for p in fb.last_profile() if p["kernel"] == "k_jkc"], default=0)
        st = fb.last_stats
        out[mode] = (f, (st.quartets_computed, st.quartets_screened, st.prim_quartets))
        fb.close()
    print("  largest launch", waves, "wavefronts, max |difference|", np.abs(out["0"][0] - out["2"][0]).max(), flush=True)
    assert waves > 65536
    assert out["0"][1] == out["2"][1]
    assert np.abs(out["0"][0] - out["2"][0]).max() <= 1e-11
