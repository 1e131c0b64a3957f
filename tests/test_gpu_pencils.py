"""The Lambda pencils at every Nw (one to eight wavefronts a pencil, and the one-wavefront kernel up to 256
with fewer samples than lanes), one and several points per workgroup, with angle bins: against the oracle at
1e-10 of the largest value (the suite's normwise bound), the bins adding up to the totals to 1e-13 (sums of
the same terms in another order)."""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

CASES = [(8, 16), (4, 32), (12, 64), (16, 128), (8, 256), (12, 512), (96, 512), (16, 1024), (64, 1024), (8, 2048),
         (4, 4096)]
P = dict(n=0.9, T=0.3, U=2.0, tp=-0.15)


@pytest.mark.parametrize("N,Nw", CASES)
def test_lambda(N, Nw, oracle_mod):
    from tpsc_conductivity_amd.tpsc import CondOpt

    print(f"[pencils] N = {N} Nw = {Nw}", flush=True)
    o = oracle_mod.Oracle(N, Nw, P["n"], P["T"], P["U"], tp=P["tp"], coarse_pass=False)
    assert o.solve()
    g = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False)
    g.solve()
    total = {f: g.get(f) for f in ("chijj1", "chijj2")}
    for f in total:
        assert relerr(total[f], o.get(f)) < 1e-10, f
    g.calc_chijj_vertex_corr_all_optim(N_theta_k=3)
    for f in total:
        bins = g.get(f + "_k").reshape(Nw // 2 + 1, 3)
        assert relerr(bins.sum(axis=1), total[f]) < 1e-13, f
    g.close()


@pytest.mark.parametrize("N,Nw", [(4, 256), (8, 512), (12, 512), (4, 1024), (12, 1024), (16, 2048), (8, 4096)])
def test_tau_pencils(N, Nw, oracle_mod):
    """chi0, V and what Sigma gives (mu, Tr Sigma G), pencils in pairs: odd and even counts of wedge points"""
    from tpsc_conductivity_amd.tpsc import CondOpt

    print(f"[pencils] N = {N} Nw = {Nw}", flush=True)
    o = oracle_mod.Oracle(N, Nw, P["n"], P["T"], P["U"], tp=P["tp"], coarse_pass=False)
    assert o.solve()
    g = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False)
    g.solve()
    assert relerr(g.get("chi0"), o.get("chiqw")) < 1e-10
    assert relerr(g.get("V"), o.get("V")) < 1e-10
    s = o.scalars()
    for k in ("mu", "kx0", "Usp", "Uch"):
        assert abs(g.scalar(k) - s[k]) < 1e-10 * max(1.0, abs(s[k])), k
    m = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False, precision="mixed")
    m.solve()
    for f in ("chi0", "V", "Sigma_kw"):
        assert relerr(m.get(f), g.get(f)) < 1e-6, f
    g.close()
    m.close()
