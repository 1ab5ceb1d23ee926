"""Vxc builds with little device memory: the batches are cut into smaller groups until
the group arrays fit, with the same result (1e-10, the bound of the Vxc tests: the same
terms in another order), and a device without room for one batch declines with the
session still usable.  OQPH_XC_WORKSPACE plays the device's free memory."""
import numpy as np
import pytest

from helpers import small_system
from openqp_amd import basis as B, molecules as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,nw,name,nfocks", [("6-31g", 3, "svwn5", 1), ("6-31g(d)", 7, "b3lyp", 2),
                                                  ("cc-pvtz", 2, "b3lyp5", 1)])
def test_vxc_in_small_groups(oracle, monkeypatch, basis, nw, name, nfocks):
    from openqp_amd.lib import FockBuilder, OqphError
    bas = small_system(basis, nw=nw, seed=4)
    S, _, _ = oracle.int1e(bas)
    D = B.pack_tri(M.random_density(S, 5 * nw, seed=7))
    dp = D if nfocks == 1 else np.concatenate([0.55 * D, 0.45 * D])
    fb = FockBuilder(bas)
    fb.set_xc(name, 20, 6)
    V, exc, nel = fb.vxc(dp, nfocks)
    one = fb.xc_grid_stats()["max_nb"] * 64 * 8  # phi of one point tile
    fb.close()
    for most in (4096 * one, 512 * one, 100 * one):
        monkeypatch.setenv("OQPH_XC_WORKSPACE", str(most))
        fb = FockBuilder(bas)
        fb.set_xc(name, 20, 6)
        Vs, es, ns = fb.vxc(dp, nfocks)
        err = max(np.abs(a - b).max() for a, b in zip(V, Vs))
        print("vxc in small groups", basis, nw, name, "workspace", most, "max |dV|", err, flush=True)
        assert err < 1e-10 and abs(es - exc) < 1e-10 and abs(ns - nel) < 1e-10
        monkeypatch.setenv("OQPH_XC_WORKSPACE", "64")
        fb.set_geometry(bas.xyz + 0.5)
        with pytest.raises(OqphError, match="one batch"):
            fb.vxc(dp, nfocks)
        monkeypatch.delenv("OQPH_XC_WORKSPACE")
        Vs, es, ns = fb.vxc(dp, nfocks)
        assert max(np.abs(a - b).max() for a, b in zip(V, Vs)) < 1e-10
        fb.close()
