"""Root searches on both sides of the one-workgroup limits (12288 terms for the sum rules, 6144 for mu): one term per
thread or less, a partly filled last term, just below and above each limit, in both precisions and through the
queued batch.  mu, Usp, Uch against the oracle at 1e-10 (the searches converge to 1e-13; the sums differ in order)."""
import pytest

pytestmark = pytest.mark.gpu

# nk8 (Nw + 1) terms: 102, 495, 5805, 3612, 9945, 9537, 10725, 19737
CASES = [(4, 16), (8, 32), (16, 128), (12, 128), (32, 64), (64, 16), (48, 32), (32, 128)]
P = dict(n=0.9, T=0.3, U=2.0, tp=-0.15)


@pytest.mark.parametrize("N,Nw", CASES)
def test_roots(N, Nw, oracle_mod):
    from tpsc_conductivity_amd.tpsc import CondOpt

    print(f"[search] N = {N} Nw = {Nw}", flush=True)
    o = oracle_mod.Oracle(N, Nw, P["n"], P["T"], P["U"], tp=P["tp"], coarse_pass=False)
    assert o.solve()
    s = o.scalars()
    for precision, tol in (("fp64", 1e-10), ("mixed", 1e-6)):
        g = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False, precision=precision)
        g.solve()
        for k in ("Usp", "Uch", "mu"):
            assert abs(g.scalar(k) - s[k]) < tol * max(1.0, abs(s[k])), (precision, k)
        g.close()


def test_queued_roots():
    from tpsc_conductivity_amd import capi
    from tpsc_conductivity_amd.tpsc import CondOpt

    arr = (capi.Params * len(CASES))()
    for a, (N, Nw) in zip(arr, CASES):
        a.nk0, a.Nw0, a.n, a.T, a.eta, a.tp, a.U = N, Nw, P["n"], P["T"], 0.1, P["tp"], P["U"]
        a.precision = capi.PRECISIONS["fp64"]
    out, _ = capi.solve_batch(arr, workers=1)
    for (N, Nw), r in zip(CASES, out):
        g = CondOpt(N, Nw, P["n"], P["T"], params=(P["tp"], 0.0, 0.0, P["U"]), coarse_pass=False)
        g.solve()
        assert r.status == 0 and abs(r.mu - g.scalar("mu")) < 1e-11, (N, Nw)
        g.close()
