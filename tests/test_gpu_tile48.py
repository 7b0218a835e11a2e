"""Matrix-core kernels around the edges of their tiles (32, 48 and 64 rows), dense and
diagonal V, real and complex parameters, direct links, against the oracle."""
import numpy as np
import pytest

import libheom_amd as H
from libheom_amd import configs
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [17, 31, 32, 33, 47, 48, 49, 63])
@pytest.mark.parametrize("dense_v", [True, False])
@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
def test_derivative(N, dense_v, real, dtype):
    print("tile", N, dense_v, real, dtype, flush=True)
    m = configs.random_model(N, 2, 2, 2, seed=N, dense_v=dense_v, offdiag_gamma=True,
                             complex_params=not real)
    g = H.heom_hilb(2, dtype=dtype).load(m, H.hip(0))
    o = O.Oracle(O.HILB, N, 2, n_threads=4).load(m)
    rng = np.random.default_rng(1)
    rho = rng.normal(size=g.main_size()) + 1j * rng.normal(size=g.main_size())
    ref = o.calc_diff(rho, 0.3 - 0.2j, 0.0)
    got = g.calc_diff_impl(None, np.zeros_like(ref), rho, 0.3 - 0.2j, 0.0)
    # FP32: sums of 4 N products and 8 links, 2^-24 each, of the largest element
    tol = 1e-10 if dtype == "complex128" else (4 * N + 8) * 2.0 ** -24
    assert np.abs(got - ref).max() <= tol * max(1.0, np.abs(ref).max())


@pytest.mark.parametrize("N", [33, 48])
@pytest.mark.parametrize("dense_v", [True, False])
def test_rkdp(N, dense_v):
    print("tile rkdp", N, dense_v, flush=True)
    m = configs.random_model(N, 2, 2, 1, seed=N, dense_v=dense_v)
    kw = {"dt": 0.01, "atol": 1e-10, "rtol": 1e-8}
    t = np.array([0.0, 0.02, 0.05])
    q = H.heom_hilb(1).load(m, H.hip(0))
    s = H.qme_solver(H.hip(0), q, H.rkdp())
    rho, _ = s.solve_rho_s(m["rho0"], t, kw)
    o = O.Oracle(O.HILB, N, 1, n_threads=4).load(m)
    rho_o, _, st_o, _, _ = o.solve(m["rho0"], t, O.RKDP, kw["dt"], kw["atol"], kw["rtol"])
    st = s.stats()
    assert (st["n_accepted"], st["n_rejected"]) == (st_o.n_accepted, st_o.n_rejected)
    assert np.abs(rho - rho_o).max() <= 1e-10 * max(1.0, np.abs(rho_o).max())
