"""The shared-links kernel in complex64: derivatives with real and complex couplings
against the oracle, and Dormand-Prince with the device walking through the output
times against one interval at a time (the stored FP32 derivative as k_1)."""
import ctypes

import numpy as np
import pytest
import torch

import libheom_amd as H
from libheom_amd import _capi
from oracle import oracle as O
from tests.test_gpu_split import model

pytestmark = pytest.mark.gpu


def bar(m, n_links, rho):
    """Rounding bound of one FP32 derivative: a sum of 2N products of H, one product per
    link, the damping and the delta term, and a few roundings of each coefficient, in
    complex arithmetic (2 sqrt 2 per product): n u times the largest sum of magnitudes."""
    N, depth = m["N"], m["max_depth"]
    v = max(np.abs(z["V"]).max() for z in m["noises"])
    cf, gam, delta = 0.0, 0.0, 0.0
    for z in m["noises"]:
        s, a = z["S"] @ z["phi_0"], z["A"] @ z["phi_0"]
        cf = max(cf, 2 * v * (np.abs(z["sigma"]).max() + depth * (np.abs(s) + np.abs(a)).max())
                 + depth * np.abs(z["gamma"] - np.diag(np.diag(z["gamma"]))).max())
        gam = max(gam, depth * np.abs(np.diag(z["gamma"])).max())
        delta += abs(z["s_delta"]) * (2 * v) ** 2
    total = np.abs(rho).max() * (2 * N * np.abs(m["H"]).max() + n_links * cf + gam + delta)
    return 2 ** -24 * 2 * np.sqrt(2) * (2 * N + n_links + 8) * total


# as test_gpu_split: the most links of an ADO are 9, 14 (and 12 of off-diagonal gamma),
# 30 and 10
@pytest.mark.parametrize("shape,n_links", [((3, 3, 1), 9), ((4, 3, 2), 26), ((6, 5, 1), 30),
                                           ((1, 5, 4), 10)])
@pytest.mark.parametrize("N", [4, 5, 7, 11, 12, 16])
@pytest.mark.parametrize("real", [True, False])
def test_derivative(N, shape, n_links, real):
    print("split c64", N, shape, real, flush=True)
    m = model(N, *shape, real, offdiag=shape == (4, 3, 2))
    g = H.heom_hilb(shape[2], dtype="complex64").load(m, H.hip(0))
    o = O.Oracle(O.HILB, N, shape[2], n_threads=4).load(m)
    rng = np.random.default_rng(1)
    rho = rng.normal(size=g.main_size()) + 1j * rng.normal(size=g.main_size())
    ref = o.calc_diff(rho, 1.0, 0.0)
    got = g.calc_diff_impl(None, np.zeros_like(ref), rho, 1.0, 0.0)
    assert np.abs(got - ref).max() <= bar(m, n_links, rho)


@pytest.mark.parametrize("N,shape", [(4, (2, 5, 2)), (5, (3, 4, 2)), (7, (4, 3, 2)),
                                     (12, (3, 4, 1)), (16, (2, 5, 1))])
@pytest.mark.parametrize("real", [True, False])
def test_rkdp_walk_equals_intervals(N, shape, real):
    print("split c64 rkdp", N, shape, real, flush=True)
    m = model(N, *shape, real)
    t = np.array([0.0, 0.05, 0.05, 0.12])
    kw = {"dt": 0.3, "atol": 1e-7, "rtol": 1e-5}  # the first attempt is rejected
    q = H.heom_hilb(shape[2], dtype="complex64").load(m, H.hip(0))
    a, b = (H.qme_solver(H.hip(0), q, H.rkdp()) for _ in range(2))
    rho_a = torch.from_numpy(m["rho0"]).cuda()
    rs = np.zeros((t.size, N * N), np.complex128)
    ptr = lambda x: x.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    _capi.check(_capi.load().heom_solve_dev(a._s, rho_a.data_ptr(), ptr(t), t.size, kw["dt"],
                                            kw["atol"], kw["rtol"], ptr(rs)))
    rho_b = m["rho0"].copy()
    b.solve(rho_b, t, None, kw)
    assert np.isfinite(rho_b).all()
    assert np.array_equal(rho_a.cpu().numpy(), rho_b)
    assert np.array_equal(rs[-1], rho_b[:N * N])
    assert a.stats() == b.stats()
