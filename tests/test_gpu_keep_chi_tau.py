"""chi0(q,tau) kept in the mixed path: FP32 values of an ordinary point (1e-6 of the FP64 path's, the mixed path's
bound), and those of a point whose spin enhancement has the chi0 stage run again in FP64: the FP64 path's bit
for bit, the same kernels."""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu

N, Nw = 32, 256
ORDINARY = dict(n=0.9, T=0.3, tp=-0.15, U=2.0)
ENHANCED = dict(n=0.9, T=0.1, tp=-0.15, U=4.0)


def kept(precision, point):
    from tpsc_conductivity_amd.tpsc import CondOpt

    g = CondOpt(N, Nw, point["n"], point["T"], params=(point["tp"], 0.0, 0.0, point["U"]), coarse_pass=False,
                precision=precision)
    g.keep_chi_tau(True)
    g.solve()
    fp64 = g.scalar("chi0_fp64")
    enh = 1.0 / (1.0 - g.scalar("Usp") * g.scalar("chi0max") / 2.0)
    out = g.get("chi0_tau")
    g.close()
    print(f"[chi_tau] {precision} {point}: enhancement {enh:.2f}", flush=True)
    return out, fp64


@pytest.mark.parametrize("point,promoted", [(ORDINARY, False), (ENHANCED, True)])
def test_kept_chi_tau(point, promoted):
    ref, _ = kept("fp64", point)
    val, fp64 = kept("mixed", point)
    assert fp64 == float(promoted)
    if promoted:
        assert np.array_equal(val, ref)
    else:
        assert relerr(val, ref) < 1e-6
