"""The cooperative J/K kernel (k_jkc) against the oracle (|f - f_oracle| <=
1e-10, the same quartet counts) and against the kernels it replaces (1e-12):
every class that has one (OQPH_JKC=2), the default choice, and none
(OQPH_JKC=0).  One water leaves most lane groups of a wavefront empty, two and
three waters give partial ones; pure and Cartesian d and f; the open-shell
pass; a range-separated build; a rank's share."""
import os
import sys

import numpy as np
import pytest

from helpers import density_for, small_system
from openqp_amd import basis as B

pytestmark = pytest.mark.gpu
TOL = 1e-10


@pytest.fixture(scope="module")
def L():
    from openqp_amd import lib
    return lib


@pytest.mark.parametrize("basis,nw,harmonic", [("6-31g", 2, None), ("6-31g(d)", 1, None), ("6-31g(d)", 3, None),
                                               ("cc-pvdz", 2, 0), ("cc-pvtz", 1, None), ("cc-pvtz", 1, 0),
                                               ("cc-pvtz", 2, None)])
def test_cooperative_kernel(L, oracle, monkeypatch, basis, nw, harmonic):
    print("k_jkc", basis, nw, harmonic, flush=True)
    bas = small_system(basis, nw=nw, seed=5)
    if harmonic is not None:
        bas = B.build_basis(basis, bas.zn.astype(int), bas.xyz, harmonic=harmonic)
    _, dp = density_for(oracle, bas, 5 * nw, seed=8)
    _, da = density_for(oracle, bas, 5 * nw, seed=9)
    da, db = 0.5 * da, 0.5 * dp
    fo, so = oracle.fock_jk(bas, dp)
    ra, rb, su = oracle.fock_jk_uhf(bas, da, db)
    out, kinds = {}, {}
    for mode in ("0", "1", "2"):
        monkeypatch.setenv("OQPH_JKC", mode)
        fb = L.FockBuilder(bas)
        f = fb.fock_jk(dp)
        st = (fb.last_stats.quartets_computed, fb.last_stats.quartets_screened, fb.last_stats.prim_quartets)
        kinds[mode] = {p["kernel"] for p in fb.last_profile()}
        fa, fbb = fb.fock_jk_uhf(da, db)
        nu = fb.last_stats.quartets_computed
        cam = fb.fock_jk_cam(dp, 0.19, 0.46, 0.33)
        fb.set_share(1, 3)
        out[mode] = (f, fa, fbb, cam, fb.fock_jk(dp))
        err = np.abs(f - fo).max()
        eu = max(np.abs(fa - ra).max(), np.abs(fbb - rb).max())
        print("  OQPH_JKC", mode, "max |f - f_oracle| =", err, "UHF", eu, sorted(kinds[mode]), flush=True)
        assert err <= TOL and eu <= TOL
        assert st[0] == int(so[1]) and nu == int(su[1])
        out[mode + "st"] = st
        fb.close()
    assert "k_jkc" not in kinds["0"] and "k_jkc" in kinds["2"]
    for mode in ("1", "2"):
        assert out[mode + "st"] == out["0st"]
        for a, b in zip(out["0"], out[mode]):
            assert np.abs(a - b).max() <= 1e-12


def test_split_primitives_bra_longer_than_the_lds_copy(L, oracle):
    """Bra-row kernels with more primitive pairs than their LDS copy holds
    (12 x 12 = 144 > 128: no splitting) next to split ones (36, 9, 1)."""
    bas = small_system("6-31g", nw=2, seed=3)
    # the two oxygens' 1s with each primitive doubled (half the coefficient): 12 primitives
    ex, cc, npr, poff = [], [], [], []
    for s in range(bas.nsh):
        e = bas.ex[bas.poff[s]:bas.poff[s] + bas.nprim[s]]
        c = bas.cc[bas.poff[s]:bas.poff[s] + bas.nprim[s]]
        if bas.nprim[s] == 6:
            e, c = np.repeat(e, 2), np.repeat(c, 2) / 2.0
        poff.append(len(ex))
        npr.append(len(e))
        ex.extend(e)
        cc.extend(c)
    big = B.Basis(bas.name, bas.am, bas.harmonic, bas.atom, np.asarray(npr, np.int32), np.asarray(poff, np.int32),
                  bas.aooff, np.asarray(ex), np.asarray(cc), bas.xyz, bas.zn)
    _, dp = density_for(oracle, big, 10, seed=4)
    fo, so = oracle.fock_jk(big, dp)
    fb = L.FockBuilder(big)
    f = fb.fock_jk(dp)
    assert np.abs(f - fo).max() <= TOL
    assert fb.last_stats.quartets_computed == int(so[1])
    fb.close()
