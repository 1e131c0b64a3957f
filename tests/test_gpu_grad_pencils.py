"""The Lambda tangent pencil at every Nw that it is compiled for (fewer samples than threads up to four per
thread): the gradient of sum_{n <= 8} Lambda_jj(iq_n), dmu/dp and d Lambda_jj(iq_n)/dp for every n against central
differences (h = 1e-5) of the oracle, at the 1e-6 of the other gradient tests."""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

H = 1e-5
LAM = 8
P = dict(n=0.9, T=0.2, U=2.0, tp=-0.15)


@pytest.mark.parametrize("N,Nw", [(8, 16), (12, 32), (8, 64), (16, 128), (12, 256), (8, 512), (16, 1024)])
def test_lambda_gradient(N, Nw, oracle_mod):
    from tpsc_conductivity_amd.tpsc import CondOpt

    print(f"[gradpencil] N = {N} Nw = {Nw}", flush=True)
    g = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False, t=1.0)
    theta = np.array([1.0, P["tp"], g.scalar("mu0"), P["U"]])
    g.fix_mu0(theta[2])
    g.loss_forward(None, LAM)
    grad = g.loss_backward(1.0)
    dmu, dlam = g.get("grad_dmu"), g.get("grad_dlambda").reshape(4, -1)
    g.close()
    fg, fmu, flam = np.zeros(4), np.zeros(4), []
    for i in range(4):
        v = []
        for sgn in (1, -1):
            t, tp, mu0, U = theta + sgn * H * np.eye(4)[i]
            o = oracle_mod.Oracle(N, Nw, P["n"], P["T"], U, tp=tp, coarse_pass=False, t=t, mu0=mu0)
            L = o.loss(None, LAM)
            v.append((L, o.scalars()["mu"], o.get("chijj1") + o.get("chijj2")))
        fg[i], fmu[i] = (v[0][0] - v[1][0]) / (2 * H), (v[0][1] - v[1][1]) / (2 * H)
        flam.append((v[0][2] - v[1][2]) / (2 * H))
    for a, b, what in ((grad, fg, "gradient"), (dmu, fmu, "dmu")):
        r = np.abs(a - b) / np.maximum(np.abs(b), 1e-3 * np.abs(b).max())
        print(f"[gradpencil] {what} {a} differences {b} rel {r}", flush=True)
        assert np.all(r < 1e-6), what
    for p in range(4):
        assert relerr(dlam[p], flam[p]) < 1e-6, p
