"""The Aslamazov-Larkin pencils on both sides of their switches (Nw = 512: half of the pencils in registers, 1024: all),
even and odd boson frequencies up to the largest: against the oracle at 1e-10 of the largest value (the bound of the
other Aslamazov-Larkin tests)."""
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,Nw,mmin", [(8, 16, 0), (8, 64, 1), (12, 512, 2), (8, 1024, 1), (4, 2048, 3)])
def test_al(N, Nw, mmin, oracle_mod):
    from tpsc_conductivity_amd.tpsc import CondOpt

    print(f"[al pencils] N = {N} Nw = {Nw}", flush=True)
    o = oracle_mod.Oracle(N, Nw, 0.9, 0.3, 2.0, tp=-0.15, coarse_pass=False)
    assert o.solve()
    o.calc_chijj(1)
    o.calc_chijj_al(mmin, 1)
    g = CondOpt(N, Nw, 0.9, 0.3, params=(-0.15, 0.0, 0.0, 2.0), coarse_pass=False)
    g.solve()
    g.calc_chijj_vertex_corr_all_optim(chi3=True, mmin=mmin)
    assert relerr(g.get("chijj3"), o.get("chijj3")) < 1e-10
    g.close()
