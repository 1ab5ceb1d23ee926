"""The dense form of the response pass (integrals stored, then matrix products)
against the per-quartet digestion (OQPH_RESPONSE=0) and the oracle: 1e-10, the
bound of the response tests; the same quartet and primitive counts.  Numbers of
densities around the 16, 32 and 64 columns of a product, with no, some and only
Coulomb components; AO counts that are no multiple of 16 or 32; s and p, Cartesian
and pure d and f; a rank's share; exchange or Coulomb alone."""
import numpy as np
import pytest

from helpers import small_system
from openqp_amd import basis as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,nw,harmonic,nmat,nf,ncoul,se,sc",
                         [("6-31g", 1, None, 1, 1, 0, 1.0, 1.0), ("6-31g", 3, None, 4, 4, 4, 0.8, 0.9),
                          ("6-31g(d)", 1, None, 7, 5, 4, 1.0, 1.0), ("cc-pvdz", 2, 0, 7, 3, 6, 0.0, 1.0),
                          ("cc-pvtz", 1, None, 1, 17, 1, 1.0, 0.0), ("cc-pvtz", 1, 0, 13, 5, 4, 0.7, 0.7)])
def test_dense_response(oracle, monkeypatch, basis, nw, harmonic, nmat, nf, ncoul, se, sc):
    from openqp_amd import lib as L
    print("dense response", basis, nw, harmonic, nmat, nf, ncoul, se, sc, flush=True)
    bas = small_system(basis, nw=nw, seed=5)
    if harmonic is not None:
        bas = B.build_basis(basis, bas.zn.astype(int), bas.xyz, harmonic=harmonic)
    rng = np.random.default_rng(3)
    n = bas.nbf
    d3 = 0.1 * np.einsum("ikcv,jkcv->ijcv", rng.standard_normal((n, 3, nmat, nf)), rng.standard_normal((n, 3, nmat, nf)))
    d3 = np.ascontiguousarray(d3)
    out = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("OQPH_RESPONSE", mode)
        fb = L.FockBuilder(bas)
        f = fb.mrsf_int2(d3, ncoul=ncoul, se=se, sc=sc)
        st = fb.last_stats
        counts = (st.quartets_computed, st.quartets_screened, st.prim_quartets)
        again = fb.mrsf_int2(-2.0 * d3, ncoul=ncoul, se=se, sc=sc)
        assert np.abs(again + 2.0 * f).max() <= 1e-9  # the coarser screen of a larger density keeps more
        fb.set_share(1, 3)
        out[mode] = (f, fb.mrsf_int2(d3, ncoul=ncoul, se=se, sc=sc), counts)
        fb.close()
    assert out["0"][2] == out["1"][2]
    for a, b in zip(out["0"][:2], out["1"][:2]):
        assert np.abs(a - b).max() <= 1e-10
    fo, so = oracle.mrsf_int2(bas, d3, ncoul=ncoul, se=se, sc=sc)
    print("  max |f - f_oracle| =", np.abs(out["1"][0] - fo).max(), "modes", np.abs(out["0"][0] - out["1"][0]).max(), flush=True)
    assert np.abs(out["1"][0] - fo).max() <= 1e-10
    assert out["1"][2][0] == so[1]
