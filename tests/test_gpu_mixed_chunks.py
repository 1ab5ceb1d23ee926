"""Which quartets of a mixed build run in FP32: 64 consecutive kets of a bra's list
together, when the bounds of all of them are below the cutoff.  The rule is the same
whether one lane evaluates a ket (the wavefront-task kernel, OQPH_JK_ROWS=0) or
several do (the bra-row kernel, which spreads the kets of a short list over idle
lanes), so both report the same count; the grouped kernel decides for all bras of a
group at once and can only keep more of them in FP64.  Counts are integers: equal
exactly."""
import pytest

from helpers import density_for
from openqp_amd import basis as B, molecules as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("basis,nw,cut", [("6-31g", 2, 1e-3), ("6-31g", 4, 1e-3), ("6-31g(d)", 3, 1e-4),
                                          ("cc-pvdz", 2, 1e-3), ("cc-pvdz", 4, 1e-5)])
def test_fp32_share_does_not_depend_on_the_kernel(oracle, monkeypatch, basis, nw, cut):
    from openqp_amd import lib as L
    print("FP32 share", basis, nw, cut, flush=True)
    Z, xyz = M.water_grid(nw, 1, 1, seed=1)
    bas = B.build_basis(basis, Z, xyz)
    _, dp = density_for(oracle, bas, 5 * nw, seed=11)
    monkeypatch.setenv("OQPH_JKC", "0")  # FP64 only, where it is used
    n = {}
    for rows, grouped in (("0", "0"), ("2", "0"), ("2", "2")):
        monkeypatch.setenv("OQPH_JK_ROWS", rows)
        monkeypatch.setenv("OQPH_JKG", grouped)
        fb = L.FockBuilder(bas, precision=1, fp32_cutoff=cut)
        fb.fock_jk(dp)
        n[rows + grouped] = fb.last_stats.quartets_fp32
        assert 0 < n[rows + grouped] < fb.last_stats.quartets_computed
        fb.close()
    print("  FP32 quartets", n, flush=True)
    assert n["20"] == n["00"]
    assert n["22"] <= n["20"]
