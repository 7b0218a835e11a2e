"""The seven passes over the state of a Dormand-Prince attempt with the projection
of rho_0: the first evaluates the operator and forms the next stage input at once."""
import ctypes

import numpy as np
import pytest

import libheom_amd as H
from libheom_amd import _capi, configs

pytestmark = pytest.mark.gpu


def stage_bytes(q, m):
    s = H.qme_solver(H.hip(0), q, H.rkdp())
    s.solve_rho_s(m["rho0"], np.array([0.0, 0.1]), {"dt": 0.1, "atol": 1e-9, "rtol": 1e-6})
    b, n = np.zeros(8), ctypes.c_int()
    _capi.check(_capi.load().heom_solver_stage_bytes(
        s._s, b.ctypes.data_as(ctypes.c_void_p), ctypes.byref(n)))
    return b[:n.value]


# real bytes per element of y, D and a stage input in complex128 and complex64
@pytest.mark.parametrize("dtype,half", [("complex128", 16), ("complex64", 8)])
def test_projected_attempt_forms_the_input_in_stage_0(dtype, half):
    m = configs.random_model(7, 2, 2, 3, seed=3, dense_v=False)
    plain, proj = (stage_bytes(H.heom_hilb(3, dtype=dtype, renorm_rho0=p).load(m, H.hip(0)), m)
                   for p in (False, True))
    n = m["rho0"].size
    assert plain.size == proj.size == 7
    assert plain[0] == (16 + 2 * half) * n
    # operator tables aside: y and (complex64) its FP32 copy read, D and the input written
    tables = proj[1] - (16 + 4 * half) * n  # stage 1 moves its input, y, D, k_2, the next input
    assert proj[0] == tables + (16 + 2 * half + (half if half == 8 else 0)) * n
    assert np.array_equal(plain[1:], proj[1:])
