"""Stages called on a sub-lattice between full solves: the buffers hold the sub-lattice too, and a full solve
afterwards gives its first values bit for bit (the solve is deterministic)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = dict(n=0.9, T=0.2, params=(-0.15, 0.0, 0.0, 2.0), coarse_pass=False)


def test_lambda_on_a_sub_lattice_with_more_workgroups():
    """64^2 (1023 points) takes 1023 workgroups, the context's 96^2 (2303 points) 768"""
    from tpsc_conductivity_amd.tpsc import CondOpt

    print("[sub-lattice] 96 x 512, Lambda on 64 x 512", flush=True)
    g = CondOpt(96, 512, P["n"], P["T"], params=P["params"], coarse_pass=False)
    g.solve()
    first = {f: g.get(f) for f in ("chijj1", "chijj2")}
    g.calc_chiqw_FFT_spline(64, 512)
    g.calc_chijj_vertex_corr_all_optim()
    g.solve()
    for f in first:
        assert np.array_equal(g.get(f), first[f]), f
    g.close()


def test_angle_bins_of_two_lattices():
    """the same number of bins on a sub-lattice first: the full lattice's bins are its own"""
    from tpsc_conductivity_amd.tpsc import CondOpt

    print("[sub-lattice] 32 x 64, 3 bins on 16 x 64 first", flush=True)
    ref = CondOpt(32, 64, P["n"], P["T"], params=P["params"], coarse_pass=False)
    ref.solve()
    ref.calc_chijj_vertex_corr_all_optim(N_theta_k=3)
    g = CondOpt(32, 64, P["n"], P["T"], params=P["params"], coarse_pass=False)
    g.solve()
    g.calc_chiqw_FFT_spline(16, 64)
    g.calc_chijj_vertex_corr_all_optim(N_theta_k=3)
    g.solve()
    g.calc_chijj_vertex_corr_all_optim(N_theta_k=3)
    for f in ("chijj1_k", "chijj2_k"):
        assert np.array_equal(g.get(f), ref.get(f)), f
    ref.close()
    g.close()


def test_local_green_function_of_two_grids():
    """fewer frequencies first: the buffer holds the full grid's"""
    from tpsc_conductivity_amd.tpsc import CondOpt

    print("[sub-lattice] 16 x 256, G_loc on 16 x 64 first", flush=True)
    ref = CondOpt(16, 256, P["n"], P["T"], params=P["params"], coarse_pass=False)
    ref.solve()
    g = CondOpt(16, 256, P["n"], P["T"], params=P["params"], coarse_pass=False)
    g.solve()
    g.calc_chiqw_FFT_spline(16, 64)
    g.Gwn_local()
    g.solve()
    assert np.array_equal(g.Gwn_local(), ref.Gwn_local())
    ref.close()
    g.close()
