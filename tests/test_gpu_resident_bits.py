"""The resident fixed-step launches give the bits of the stage kernels where the
parameters are real (up to five levels: the kernels without per-noise tables)."""
import numpy as np
import pytest

import libheom_amd as H
from libheom_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["rk4", "lsrk4"])
@pytest.mark.parametrize("K", [1, 2, 4])
@pytest.mark.parametrize("N", [2, 3, 4, 5])
def test_resident_bits_equal_stage_kernels(N, K, method):
    m = configs.random_model(N, 1, K, 2, seed=10 * N + K, dense_v=False, complex_params=False)
    eng = H.hip(0)
    q = H.heom_hilb(2).load(m, eng)
    assert q.main_size() <= 1024
    out = []
    for resident in (True, False):
        s = H.qme_solver(eng, q, getattr(H, method)())
        s.set_graphs(resident)
        out.append(s.solve_rho_s(m["rho0"], np.array([0.0, 0.105, 0.2]), {"dt": 0.01}))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
