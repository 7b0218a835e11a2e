"""The kernel that shares an ADO's links between groups of lanes, against the
oracle: every block size, real and complex couplings, links beyond one round,
units with idle groups, and both drivers."""
import numpy as np
import pytest

import libheom_amd as H
from libheom_amd import configs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-10


def model(N, n_noise, ln, L, real, offdiag=False):
    m = configs.random_model(N, n_noise, ln, L, seed=10 * N + L, dense_v=False,
                             offdiag_gamma=offdiag, complex_params=not real)
    if not real:  # complex diagonals of V
        rng = np.random.default_rng(N)
        for z in m["noises"]:
            z["V"] = z["V"] + 1j * np.diag(rng.normal(size=N))
    return m


# (noises, modes per noise, depth): 9 links at the root and 1 at the other ADOs,
# 12 + 2, 30 at the root (two rounds of the shared ADO), 5 + 4
@pytest.mark.parametrize("shape", [(3, 3, 1), (4, 3, 2), (6, 5, 1), (1, 5, 4)])
@pytest.mark.parametrize("N", list(range(4, 17)))
@pytest.mark.parametrize("real", [True, False])
def test_derivative(N, shape, real):
    print("split", N, shape, real, flush=True)
    m = model(N, *shape, real, offdiag=shape == (4, 3, 2))
    g = H.heom_hilb(shape[2]).load(m, H.hip(0))
    o = O.Oracle(O.HILB, N, shape[2], n_threads=4).load(m)
    rng = np.random.default_rng(1)
    rho = rng.normal(size=g.main_size()) + 1j * rng.normal(size=g.main_size())
    ref = o.calc_diff(rho, 0.3 - 0.2j, 0.0)
    got = g.calc_diff_impl(None, np.zeros_like(ref), rho, 0.3 - 0.2j, 0.0)
    assert np.abs(got - ref).max() <= TOL * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("N,shape", [(4, (2, 5, 2)), (5, (3, 4, 2)), (7, (4, 3, 2)),
                                     (12, (3, 4, 1))])
@pytest.mark.parametrize("solver", ["rk4", "rkdp"])
def test_solve(N, shape, solver):
    print("split solve", N, shape, solver, flush=True)
    m = model(N, *shape, True)
    t = np.array([0.0, 0.05, 0.12])
    kw = {"dt": 0.02} if solver == "rk4" else {"dt": 0.02, "atol": 1e-10, "rtol": 1e-8}
    q = H.heom_hilb(shape[2]).load(m, H.hip(0))
    s = H.qme_solver(H.hip(0), q, H.rk4() if solver == "rk4" else H.rkdp())
    rho, rs = s.solve_rho_s(m["rho0"], t, kw)
    o = O.Oracle(O.HILB, N, shape[2], n_threads=4).load(m)
    rho_o, rs_o, st_o, _, _ = o.solve(m["rho0"], t, O.RK4 if solver == "rk4" else O.RKDP,
                                      kw["dt"], kw.get("atol", 0.0), kw.get("rtol", 0.0))
    scale = max(1.0, np.abs(rho_o).max())
    assert np.abs(rho - rho_o).max() <= TOL * scale
    if solver == "rkdp":
        st = s.stats()
        assert (st["n_accepted"], st["n_rejected"]) == (st_o.n_accepted, st_o.n_rejected)
