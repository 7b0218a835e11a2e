"""Long runs replay their launches from HIP graphs: the results equal, to the last bit,
those of the same launches made one by one, at every output, over runs with several graph
sizes and remainders, with outputs, host copies and changes of the operator in between."""
import numpy as np
import pytest

import libheom_amd as H
from libheom_amd import _capi, configs
from libheom_amd import closure as C

pytestmark = pytest.mark.gpu


def runs(q, m, method, t, kw, change=None):
    """State, rho_S and counters of solve_rho_s, and the states a callback sees."""
    eng = H.hip(0)
    out = []
    for graphs in (False, True):
        if change:
            q.load(m, eng)
        s = H.qme_solver(eng, q, getattr(H, method)())
        s.set_graphs(graphs)
        rho, rs = s.solve_rho_s(m["rho0"], t, kw)
        host, seen = m["rho0"].copy(), []

        def cb(tt):
            seen.append(host.copy())
            if change and len(seen) == t.size // 2:
                change(q, m, eng)

        s.reset()
        s.solve(host, t, cb, kw)
        st = s.stats()
        out.append((rho, np.asarray(rs), np.array(seen), host, st))
    (a, b) = out
    assert np.isfinite(a[0]).all()
    for x, y in zip(a[:4], b[:4]):
        assert np.array_equal(x, y)
    assert a[4] == b[4]
    if not change:  # the two entry points agree as well
        assert np.array_equal(b[0], b[3])
    return b[4]


def scaled(N, dep, seed, **kw):
    m = configs.random_model(N, 2, 2, dep, seed=seed, dense_v=False, **kw)
    m["H"] = 0.2 * m["H"]
    assert m["rho0"].size > 1024  # larger than the resident launches take
    return m


# steps per interval: several graphs and a remainder in every interval (31 = 3 x 8 + 7), one
# interval longer than all graphs, and few intervals with a remainder
@pytest.mark.parametrize("steps,n_int", [(31, 18), (600, 1), (203, 3)])
@pytest.mark.parametrize("method,dtype,proj", [("rk4", "complex128", False),
                                               ("lsrk4", "complex64", False),
                                               ("rk4", "complex64", True)])
def test_fixed_steps(method, dtype, proj, steps, n_int):
    print("replay", method, dtype, proj, steps, n_int, flush=True)
    m = scaled(5, 4, 5)
    q = H.heom_hilb(4, dtype=dtype, renorm_rho0=proj).load(m, H.hip(0))
    dt = 1e-3
    t = dt * (steps + 0.5) * np.arange(n_int + 1)
    st = runs(q, m, method, t, {"dt": dt})
    assert st["n_attempts"] >= n_int * (steps + 1)


# the shortest intervals replay graphs of 2 and 4 steps; 8 replays of them are the fewest
@pytest.mark.parametrize("steps,n_int", [(2, 9), (3, 8), (4, 12), (7, 8), (9, 8), (65, 1)])
@pytest.mark.parametrize("dtype,proj", [("complex128", False), ("complex64", True)])
def test_short_intervals(dtype, proj, steps, n_int):
    print("replay short", dtype, proj, steps, n_int, flush=True)
    m = scaled(5, 4, 6)
    q = H.heom_hilb(4, dtype=dtype, renorm_rho0=proj).load(m, H.hip(0))
    t = 1e-3 * (steps + 0.5) * np.arange(n_int + 1)
    st = runs(q, m, "rk4", t, {"dt": 1e-3})
    assert st["n_attempts"] == n_int * (steps + 1)


# above 65 536 elements eight times the replays are asked for
def test_large_hierarchy():
    m = configs.random_model(7, 3, 4, 4, seed=3, dense_v=False, complex_params=False)
    assert 1 << 16 < m["rho0"].size <= 1 << 17
    q = H.heom_hilb(4).load(m, H.hip(0))
    runs(q, m, "rk4", 1e-4 * 24.5 * np.arange(26), {"dt": 1e-4})


@pytest.mark.parametrize("N,dep,dtype,proj",
                         [(3, 5, "complex128", False), (5, 4, "complex64", False),
                          (7, 3, "complex128", True), (18, 3, "complex64", False)])
def test_dormand_prince(N, dep, dtype, proj):
    print("replay rkdp", N, dtype, proj, flush=True)
    m = scaled(N, dep, N, complex_params=False)
    q = H.heom_hilb(dep, dtype=dtype, renorm_rho0=proj).load(m, H.hip(0))
    t = 2.0 * np.array([0.0, 0.5, 0.5, 1.0, 1.5])
    kw = {"dt": 0.01, "atol": 1e-13, "rtol": 1e-12 if dtype == "complex128" else 1e-9}
    st = runs(q, m, "rkdp", t, kw)
    assert st["n_attempts"] > 200


def test_batch():
    ms = configs.batched_sweep(n_inst=5, seed=9, n_steps=600, out_every=200)
    b = H.heom_batch([H.heom_hilb(m["max_depth"]).load(m, H.hip(0)) for m in ms])
    rho0 = b.pack([m["rho0"] for m in ms])
    out = []
    for graphs in (False, True):
        s = H.qme_solver(H.hip(0), b, H.rk4())
        s.set_graphs(graphs)
        out.append(s.solve_rho_s(rho0, ms[0]["t_list"], {"dt": ms[0]["dt"]}))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("method", ["rk4", "rkdp"])
def test_operator_changed_between_replays(method):
    m = scaled(5, 4, 8, complex_params=False)
    q = H.heom_hilb(4).load(m, H.hip(0))

    def change(q, m, eng):
        q.H = 1.5 * m["H"]
        q.set_param(eng)

    if method == "rk4":
        runs(q, m, method, 0.3 * np.arange(5), {"dt": 1e-3}, change)
    else:
        runs(q, m, method, 0.5 * np.arange(5), {"dt": 0.01, "atol": 1e-13, "rtol": 1e-12}, change)


def test_closure_bound_between_replays():
    m = scaled(4, 4, 4, complex_params=False)
    q = H.heom_hilb(4).load(m, H.hip(0))
    _, n_in, n_out = C.dims(q, _capi.HEOM_CLOSURE_PER_ADO, 0)
    net = C.Mlp(n_in, 32, n_out, seed=3)
    runs(q, m, "rk4", 0.3 * np.arange(5), {"dt": 1e-3}, lambda q, m, eng: q.set_closure(net))
