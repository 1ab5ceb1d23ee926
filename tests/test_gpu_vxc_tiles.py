"""The grouped Vxc kernels against the oracle (1e-10, the bound of the Vxc tests)
where a tile can go wrong: grids of a few points (tiles and parts partly filled),
function counts around the 16, 32, 64 and 128 columns of a pass, f shells, pure and
Cartesian, LDA and GGA, one and two spins."""
import numpy as np
import pytest

from helpers import small_system
from openqp_amd import basis as B, molecules as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,nw,harmonic,name,nfocks,nrad,ntheta",
                         [("6-31g", 1, None, "b3lyp5", 1, 3, 2), ("6-31g", 1, None, "svwn5", 2, 7, 3),
                          ("6-31g", 5, None, "blyp", 1, 12, 4), ("6-31g(d)", 7, None, "b3lyp", 2, 9, 4),
                          ("cc-pvdz", 2, 0, "bhhlyp", 1, 15, 5), ("cc-pvtz", 1, None, "b3lyp5", 2, 21, 6),
                          ("cc-pvtz", 1, 0, "slater", 1, 14, 5), ("cc-pvtz", 2, 0, "b3lyp5", 1, 8, 3)])
def test_vxc_tiles(oracle, basis, nw, harmonic, name, nfocks, nrad, ntheta):
    from openqp_amd.lib import FockBuilder
    from oracle import xc as X
    print("vxc tiles", basis, nw, harmonic, name, nfocks, nrad, ntheta, flush=True)
    bas = small_system(basis, nw=nw, seed=4)
    if harmonic is not None:
        bas = B.build_basis(basis, bas.zn.astype(int), bas.xyz, harmonic=harmonic)
    S, _, _ = oracle.int1e(bas)
    D = M.random_density(S, 5 * nw, seed=7)
    dens = D if nfocks == 1 else [0.55 * D, 0.45 * D]
    dp = B.pack_tri(D) if nfocks == 1 else np.concatenate([B.pack_tri(x) for x in dens])
    fb = FockBuilder(bas)
    fb.set_xc(name, nrad, ntheta)
    V, exc, nel = fb.vxc(dp, nfocks)
    pts, w, _ = X.molecular_grid(bas.zn, bas.xyz, nrad, ntheta)
    Vo, exco, nelo = X.vxc(bas, dens, name, (pts, w), oracle, nfocks)
    for s in range(nfocks):
        err = np.abs(B.unpack_tri(V[s], bas.nbf) - Vo[s]).max()
        print("  nbf", bas.nbf, "points", len(w), "spin", s, "max |dV|", err, flush=True)
        assert err < 1e-10
    assert abs(exc - exco) < 1e-10 and abs(nel - nelo) < 1e-10
    fb.close()
