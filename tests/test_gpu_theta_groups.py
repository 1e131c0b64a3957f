"""Lambda_jj by angle of k with the points of a bin spread over workgroups of one to several points: each bin
against the oracle at 1e-10 of the largest total (the suite's normwise bound), on pencils of one wavefront with idle
lanes, of one and of several wavefronts; more bins than points, so that some are empty; and the memory of
the call, which grows with the points and not with points times bins."""
import ctypes

import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

P = dict(n=0.9, T=0.3, U=2.0, tp=-0.15)
# points per workgroup: 1 (3, 143, 63 points), 3 (2303), 4 (4095)
CASES = [(4, 16, 64), (24, 64, 7), (16, 1024, 16), (8, 2048, 5), (96, 256, 5), (96, 1024, 3), (128, 128, 64)]


@pytest.mark.parametrize("N,Nw,nth", CASES)
def test_bins_match_oracle(N, Nw, nth, oracle_mod):
    from tpsc_conductivity_amd.tpsc import CondOpt

    print(f"[theta] N = {N} Nw = {Nw} bins = {nth}", flush=True)
    o = oracle_mod.Oracle(N, Nw, P["n"], P["T"], P["U"], tp=P["tp"], coarse_pass=False)
    assert o.solve()
    o.calc_chijj(nth)
    g = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False)
    g.solve()
    one = {f: g.get(f) for f in ("chijj1", "chijj2")}
    sc = {k: g.scalar(k) for k in ("kx0", "chijj1_inf2", "chijj2_inf2", "chijj2_inf4")}
    g.calc_chijj_vertex_corr_all_optim(N_theta_k=nth)
    for f in one:
        a, b = g.get(f + "_k"), o.get(f + "_k")
        assert a.size == (Nw // 2 + 1) * nth
        assert float(np.abs(a - b).max() / np.abs(o.get(f)).max()) < 1e-10, f
        assert relerr(a.reshape(-1, nth).sum(axis=1), one[f]) < 1e-13, f
    for k, v in sc.items():  # the same terms in another order
        assert abs(g.scalar(k) - v) <= 1e-12 * max(1.0, abs(v)), k
    g.close()


@pytest.mark.parametrize("N,Nw", [(32, 256), (64, 512)])
def test_binned_memory(N, Nw):
    from tpsc_conductivity_amd import capi
    from tpsc_conductivity_amd.tpsc import CondOpt

    g = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False)
    g.solve()
    use = []
    for nth in (1, 64):
        g.calc_chijj_vertex_corr_all_optim(N_theta_k=nth)
        d = ctypes.c_double()
        capi.lib().tpsc_device_bytes(g.ctx.handle, ctypes.byref(d))
        use.append(d.value)
    nq = (N // 2 + 1) * (N // 2 - 1)
    # a pair of rows per point and per bin, the four sums of a workgroup, the tables of the bins
    rows = 2 * (Nw // 2 + 1) * 8
    print(f"[theta] {N} x {Nw}: {use[1] - use[0]:.0f} bytes for 64 bins", flush=True)
    assert use[1] - use[0] <= (nq + 2 * 64) * (rows + 4 * 8) + 64 * 1024
    g.close()
