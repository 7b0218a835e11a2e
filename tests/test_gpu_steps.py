"""Dormand-Prince attempts with the step pass between them: the device walking
through the output times (heom_solve_dev) against one interval at a time
(heom_solve) and the oracle, with intervals of no length, rejections, and more
error-norm partials than the step pass reads in one launch."""
import ctypes

import numpy as np
import pytest
import torch

import libheom_amd as H
from libheom_amd import _capi, configs
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-10


def solve_dev(s, rho0, t, kw):
    rho = torch.from_numpy(rho0).cuda()
    t = np.ascontiguousarray(t)
    rs = np.zeros((t.size, s.qme.n_level ** 2), np.complex128)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    _capi.check(_capi.load().heom_solve_dev(s._s, rho.data_ptr(), ptr(t), t.size, kw["dt"],
                                            kw["atol"], kw["rtol"], ptr(rs)))
    return rho.cpu().numpy(), rs, s.stats()


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("N", [3, 7, 18])
@pytest.mark.parametrize("t", [[0.0, 0.0, 0.2, 0.2, 0.2, 0.5, 0.5], [0.0, 0.4], [0.0, 0.0],
                               [0.0]])
def test_device_walk_equals_intervals(N, dtype, t):
    print("device walk", N, dtype, t, flush=True)
    eng = H.hip(0)
    m = configs.random_model(N, 2, 2, 2, seed=N, dense_v=False)
    kw = {"dt": 1.0, "atol": 1e-9, "rtol": 1e-6}
    q = H.heom_hilb(2, dtype=dtype).load(m, eng)
    a, b = (H.qme_solver(eng, q, H.rkdp()) for _ in range(2))
    b.set_graphs(False)  # the stage kernels also where a resident launch would do
    a.set_graphs(False)
    for _ in range(2):  # the second solve starts from the first one's step size
        rho_a, rs_a, st_a = solve_dev(a, m["rho0"], t, kw)
        rho_b, rs_b = b.solve_rho_s(m["rho0"], np.array(t), kw)
        st_b = b.stats()
        assert np.array_equal(rho_a, rho_b)
        assert np.array_equal(rs_a.reshape(-1), np.asarray(rs_b).reshape(-1))
        assert st_a == st_b
    if dtype == "complex128":
        o = O.Oracle(O.HILB, N, 2, n_threads=4).load(m)
        c = H.qme_solver(eng, q, H.rkdp())
        c.set_graphs(False)
        rho_c, rs_c, st_c = solve_dev(c, m["rho0"], t, kw)
        rho_o, rs_o, st_o, _, _ = o.solve(m["rho0"], np.array(t), O.RKDP, kw["dt"], kw["atol"],
                                          kw["rtol"])
        # the oracle's zero-length intervals differ: only lists without one
        if len(set(t)) == len(t) and len(t) > 1:
            assert st_c["n_rejected"] == st_o.n_rejected
            assert st_c["n_accepted"] == st_o.n_accepted
            scale = max(1.0, np.abs(rho_o).max())
            assert np.abs(rho_c - rho_o).max() <= TOL * scale


def test_more_partials_than_one_launch_reads():
    """33 649 ADOs of 6x6, one partial each: the decision in a launch of its own."""
    m = configs.random_model(6, 3, 6, 5, seed=2, dense_v=False)
    eng = H.hip(0)
    q = H.heom_hilb(5).load(m, eng)
    assert q.n_hrchy == 33649
    kw = {"dt": 0.02, "atol": 1e-10, "rtol": 1e-8}
    t = np.array([0.0, 0.03, 0.05])
    rho, rs, st = solve_dev(H.qme_solver(eng, q, H.rkdp()), m["rho0"], t, kw)
    o = O.Oracle(O.HILB, 6, 5, n_threads=8).load(m)
    rho_o, rs_o, st_o, _, _ = o.solve(m["rho0"], t, O.RKDP, kw["dt"], kw["atol"], kw["rtol"])
    assert (st["n_accepted"], st["n_rejected"]) == (st_o.n_accepted, st_o.n_rejected)
    assert np.abs(rho - rho_o).max() <= TOL * max(1.0, np.abs(rho_o).max())
    assert np.abs(rs.reshape(-1) - np.asarray(rs_o).reshape(-1)).max() <= TOL
