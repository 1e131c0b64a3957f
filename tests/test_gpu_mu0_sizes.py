"""The search for mu0 keeps 1, 3 or 9 wedge points per thread (up to 1024, 3072, 9216 points): sizes on both sides
of those limits and the smallest, and fillings and temperatures whose Fermi factors run under.  The residual of the
density, summed exactly on the CPU, is at most 1e-13: about 40 roundings of sums and factors of at most 2 (2e-14), and
a last step of 1e-16 relative times n'(mu) <= 2 / (4 T)."""
import math

import pytest

pytestmark = pytest.mark.gpu


def density(N, tp, T, mu):
    """(2 / N^2) sum over the N x N zone of the Fermi factors."""
    c = [math.cos(2.0 * math.pi * i / N) for i in range(N)]
    f = []
    for a in c:
        for b in c:
            x = (-2.0 * (a + b) - 4.0 * tp * a * b - mu) / T
            f.append(math.exp(-x) / (1.0 + math.exp(-x)) if x > 0 else 1.0 / (1.0 + math.exp(x)))
    return 2.0 * math.fsum(f) / N**2


@pytest.mark.parametrize("N", [4, 16, 64, 96, 128, 192, 256])  # 6, 45, 561, 1225, 2145, 4753, 8385 points
@pytest.mark.parametrize("n,T", [(0.9, 0.3), (1.37, 0.05), (0.1, 1.0)])
def test_density(N, n, T):
    from tpsc_conductivity_amd.tpsc import CondOpt

    print(f"[mu0] N = {N} n = {n} T = {T}", flush=True)
    tp = -0.2
    g = CondOpt(N, 16, n, T, params=(tp, 0.0, 0.0, 2.0), coarse_pass=False)
    mu = g.scalar("mu0")
    g.close()
    assert abs(density(N, tp, T, mu) - n) < 1e-13
