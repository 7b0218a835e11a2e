"""Parameters changed by the callback of heom_solve: the run equals, to the last
bit, two solves with the change made between them (the second starts from the
first one's step size)."""
import numpy as np
import pytest

import libheom_amd as H
from libheom_amd import _capi, configs
from libheom_amd import closure as C

pytestmark = pytest.mark.gpu

T = np.array([0.0, 0.3, 0.3, 0.6, 0.9])
KW = {"dt": 0.05, "atol": 1e-10, "rtol": 1e-7}
AT = 2  # the output before which the change happens (t = 0.3, for the second time)


def set_h(q, m, eng):
    q.H = 1.7 * m["H"]
    q.set_param(eng)


def dense_v(q, m, eng):
    x = np.arange(m["N"] ** 2).reshape(m["N"], m["N"])
    for u in range(len(m["noises"])):
        q.V[u] = q.V[u] + 0.1 * (x + x.T)
    q.set_param(eng)


def compare(m, dtype, method, graphs, change):
    print("callback", m["name"], dtype, method, graphs, change.__name__, flush=True)
    eng = H.hip(0)
    out = []
    for piecewise in (True, False):
        q = H.heom_hilb(m["max_depth"], dtype=dtype).load(m, eng)
        s = H.qme_solver(eng, q, getattr(H, method)())
        s.set_graphs(graphs)
        rho = m["rho0"].copy()
        if piecewise:
            s.solve(rho, T[:AT + 1], None, KW)
            change(q, m, eng)
            s.solve(rho, T[AT:], None, KW)
        else:
            seen = []

            def cb(t):
                seen.append(t)
                if len(seen) == AT + 1:
                    change(q, m, eng)

            s.solve(rho, T, cb, KW)
            assert seen == list(T)
        st = s.stats()
        out.append((rho, [st[k] for k in ("n_rhs", "n_attempts", "n_accepted", "n_rejected")]))
    assert np.isfinite(out[0][0]).all()
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1] == out[1][1]


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("method", ["rkdp", "rk4", "lsrk4"])
@pytest.mark.parametrize("N", [2, 7, 18])
@pytest.mark.parametrize("graphs", [True, False])
def test_hamiltonian_changed_in_callback(N, method, dtype, graphs):
    m = configs.random_model(N, 2, 2, 2, seed=N, dense_v=False)
    compare(m, dtype, method, graphs, set_h)


@pytest.mark.parametrize("method", ["rkdp", "rk4"])
def test_dense_coupling_set_in_callback(method):
    """From a resident problem (diagonal V) to one that is not."""
    m = configs.random_model(2, 2, 2, 2, seed=5, dense_v=False)
    compare(m, "complex128", method, True, dense_v)


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("method", ["rkdp", "rk4"])
def test_closure_bound_in_callback(method, graphs):
    m = configs.random_model(4, 2, 2, 2, seed=6, dense_v=False)
    eng = H.hip(0)
    q = H.heom_hilb(m["max_depth"]).load(m, eng)
    _, n_in, n_out = C.dims(q, _capi.HEOM_CLOSURE_PER_ADO, 0)
    net = C.Mlp(n_in, 32, n_out, seed=3)

    def bind(q, m, eng):
        q.set_closure(net)

    compare(m, "complex128", method, graphs, bind)


@pytest.mark.parametrize("method", ["rkdp", "rk4"])
def test_size_changed_in_callback_is_refused(method):
    """A hierarchy that no longer fits the solver's buffers ends the solve."""
    m = configs.random_model(3, 2, 2, 2, seed=7, dense_v=False)
    eng = H.hip(0)
    q = H.heom_hilb(m["max_depth"]).load(m, eng)
    s = H.qme_solver(eng, q, getattr(H, method)())

    def cb(t):
        if t == T[1]:
            q.hrchy_filter = lambda n, depth: depth < 2
            q.set_param(eng)

    with pytest.raises(H.HeomError):
        s.solve(m["rho0"].copy(), T, cb, KW)
