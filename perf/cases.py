"""What a user of libheom_amd has it compute, as a list of measurable cases.

Each case is one call (or one short run) through the public classes or the C
ABI, on inputs made from a seed.  `listed` names twelve of them, `draw` gives
others of the same families and ranges, `prepare` builds what a program holds
before the call (parameters set up, solver or network created, initial state),
`run` makes the call, `work` counts what it cannot do without, and `exact`
gives the same results in 64 bits from plain torch / numpy.

Families (the models are the repository's own: a spin-boson system, an exciton
chain with one Drude bath per site, a dense N-level system with a few baths, a
sweep of many small systems, a four-site chain with a learned closure):

  spin_boson   heom_hilb, N = 2: the smallest hierarchies; latency and launches
  chain        heom_hilb, 5..12 sites: the headline workload and its relatives
  dense        heom_hilb, 17..64 levels, diagonal coupling operators
  dense_v      heom_hilb, 17..64 levels, dense coupling operators
  sweep        heom_batch of small systems of uneven size
  liou, ado    the Liouville-space and the global sparse form of the chain
  closure      a chain run with the truncation-closure network bound
  grad         loss and gradient of that network on a training batch
"""
import ctypes
import math

import numpy as np
import torch

import libheom_amd as H
from libheom_amd import _capi
from libheom_amd import closure as C

HBAR_CM_FS = 5308.837458876145  # hbar in cm^-1 fs
KB_CM_K = 0.69503476            # k_B in cm^-1 / K


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: 66 ADOs of 2x2, fixed steps, from host arrays
        {"name": "spin_boson_rk4", "family": "spin_boson", "depth": 10, "modes": 2,
         "method": "rk4", "dt": 0.01, "outputs": 20, "steps": 10, "entry": "solve_rho_s"},
        # the reference's own call: solve() with a callback that looks at the host state at
        # every output time, adaptive steps
        {"name": "spin_boson_rkdp", "family": "spin_boson", "depth": 6, "modes": 2,
         "method": "rkdp", "dt": 0.01, "outputs": 10, "t_out": 0.2, "rtol": 1e-8,
         "entry": "solve"},
        # the headline workload: 12 650 ADOs of 7x7, adaptive steps, state resident in HBM
        {"name": "chain7_rkdp", "family": "chain", "sites": 7, "depth": 4, "modes": 3,
         "method": "rkdp", "dt": 0.1, "outputs": 5, "t_out": 10.0, "rtol": 1e-8,
         "dtype": "complex128"},
        # an odd site count in the FP32 variant (9x9 blocks, 4 060 ADOs)
        {"name": "chain9_rkdp_c64", "family": "chain", "sites": 9, "depth": 3, "modes": 3,
         "method": "rkdp", "dt": 0.1, "outputs": 5, "t_out": 10.0, "rtol": 1e-7,
         "dtype": "complex64"},
        # large blocks: 969 ADOs of 64x64, adaptive steps, FP64
        {"name": "dense64_rkdp", "family": "dense", "levels": 64, "depth": 3, "baths": 4,
         "modes": 4, "method": "rkdp", "dt": 0.01, "outputs": 2, "t_out": 0.25, "rtol": 1e-6,
         "dtype": "complex128"},
        # a block size that is no multiple of the tile, split-bf16 products
        {"name": "dense48_rkdp_bf16x3", "family": "dense", "levels": 48, "depth": 3,
         "baths": 4, "modes": 4, "method": "rkdp", "dt": 0.01, "outputs": 2, "t_out": 0.25,
         "rtol": 1e-6, "dtype": "complex64_bf16x3"},
        # one derivative evaluation of a caller with its own integrator, dense V
        {"name": "dense_v64_diff", "family": "dense_v", "levels": 64, "depth": 3, "baths": 4,
         "modes": 4, "dtype": "complex128"},
        # parameter sweep: 512 systems of N in {2, 4, 8} and uneven depth in one batch
        {"name": "sweep512_rk4_c64", "family": "sweep", "members": 512, "dt": 0.005,
         "outputs": 2, "steps": 20, "dtype": "complex64"},
        # the other two forms of the operator on chains
        {"name": "liou7_rk4", "family": "liou", "sites": 7, "depth": 2, "modes": 3, "dt": 0.5,
         "outputs": 2, "steps": 20},
        {"name": "ado4_rk4", "family": "ado", "sites": 4, "depth": 4, "modes": 2, "dt": 0.5,
         "outputs": 2, "steps": 20},
        # truncation closure: network and operator in every stage (165 ADOs of 4x4)
        {"name": "closure4_rk4", "family": "closure", "sites": 4, "depth": 3, "modes": 2,
         "hidden": 256, "dt": 0.01, "outputs": 5, "steps": 10},
        # its training: one minibatch's loss and gradient
        {"name": "closure_grad", "family": "grad", "rows": 4096, "inputs": 49, "hidden": 256,
         "targets": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["spin_boson", "chain", "chain", "dense", "dense", "dense_v", "sweep",
                         "sweep", "liou", "ado", "closure", "grad"])
    c = {"family": family}
    if family == "spin_boson":
        c.update(depth=rng.randint(3, 12), modes=rng.randint(2, 3),
                 method=rng.choice(["rk4", "rkdp"]), dt=0.01)
        c["outputs"] = rng.randint(1, 25)
        c["entry"] = rng.choice(["solve", "solve_rho_s"])
        if c["method"] == "rk4":
            c["steps"] = _log_int(rng, 3, 40)
        else:
            c.update(t_out=rng.uniform(0.05, 0.3), rtol=10.0 ** rng.randint(-9, -6))
    elif family == "chain":
        n = rng.randint(5, 12)
        top = {5: 5, 6: 4, 7: 4}.get(n, 3)
        c.update(sites=n, depth=rng.randint(1, top), modes=rng.randint(2, 3) if top > 3 else 2,
                 method=rng.choice(["rk4", "rkdp"]), outputs=rng.randint(1, 4),
                 dtype=rng.choice(["complex128", "complex64"]))
        if c["method"] == "rk4":
            c.update(dt=0.2, steps=_log_int(rng, 3, 40))
        else:
            c.update(dt=0.1, t_out=rng.uniform(2.0, 10.0), rtol=10.0 ** rng.randint(-8, -6))
    elif family == "dense":
        c.update(levels=rng.randint(17, 64), depth=rng.randint(1, 3), baths=rng.randint(2, 4),
                 modes=rng.randint(2, 4), outputs=rng.randint(1, 2),
                 dtype=rng.choice(["complex128", "complex64", "complex64_bf16x3"]),
                 method=rng.choice(["rk4", "rkdp"]), dt=0.01)
        if c["method"] == "rk4":
            c["steps"] = _log_int(rng, 2, 12)
        else:
            c.update(t_out=rng.uniform(0.05, 0.2), rtol=10.0 ** rng.randint(-7, -5))
    elif family == "dense_v":
        c.update(levels=rng.randint(17, 64), depth=rng.randint(1, 3), baths=rng.randint(2, 4),
                 modes=rng.randint(2, 4), dtype=rng.choice(["complex128", "complex64"]))
    elif family == "sweep":
        c.update(members=_log_int(rng, 4, 400), dt=0.005, outputs=rng.randint(1, 2),
                 steps=rng.randint(3, 20), dtype=rng.choice(["complex128", "complex64"]))
    elif family in ("liou", "ado"):
        n = rng.randint(2, 7)
        c.update(sites=n, depth=rng.randint(1, 4 if n <= 4 else 2), modes=2, dt=0.5,
                 outputs=rng.randint(1, 2), steps=_log_int(rng, 3, 20))
    elif family == "closure":
        c.update(sites=rng.randint(2, 5), depth=rng.randint(2, 3), modes=2,
                 hidden=rng.choice([64, 100, 128, 256]), dt=0.01, outputs=rng.randint(1, 3),
                 steps=_log_int(rng, 3, 12))
    else:
        c.update(rows=_log_int(rng, 100, 4096), inputs=rng.randint(20, 80),
                 hidden=rng.choice([64, 100, 128, 256]), targets=rng.randint(8, 64))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _drude(lam, gam, T, n):
    """Exponents and weights of a Drude bath: the Drude pole, then n - 1
    Matsubara terms, and the white-noise residual."""
    nu, c = [gam], [lam * gam * (1.0 / math.tan(0.5 * gam / T) - 1.0j)]
    for k in range(1, n):
        v = 2.0 * math.pi * k * T
        nu.append(v)
        c.append(4.0 * lam * gam * T * v / (v * v - gam * gam))
    nu, c = np.array(nu), np.array(c, np.complex128)
    return nu, c, 2.0 * lam * T / gam - float(np.sum(c.real / nu))


def _noise(V, bath):
    nu, c, delta = bath
    n = len(nu)
    return {"V": np.asarray(V, np.complex128), "gamma": np.diag(nu).astype(np.complex128),
            "phi_0": np.ones(n, np.complex128), "sigma": np.ones(n, np.complex128),
            "S": np.diag(c.real).astype(np.complex128),
            "A": np.diag(c.imag).astype(np.complex128), "s_delta": complex(delta)}


def _chain_model(rng, n, modes, depth):
    """Exciton chain in rad/fs: site energies and couplings of 100 cm^-1, one
    Drude bath per site (35 cm^-1, 50 fs, 300 K)."""
    J = np.triu(rng.uniform(-100.0, 100.0, (n, n)), 1)
    Hm = (np.diag(rng.normal(0.0, 100.0, n)) + J + J.T) / HBAR_CM_FS
    bath = _drude(35.0 / HBAR_CM_FS, 1.0 / 50.0, KB_CM_K * 300.0 / HBAR_CM_FS, modes)
    noises = []
    for u in range(n):
        V = np.zeros((n, n))
        V[u, u] = 1.0
        noises.append(_noise(V, bath))
    return {"N": n, "H": Hm.astype(np.complex128), "noises": noises, "max_depth": depth}


def _dense_model(rng, n, baths, modes, depth, dense_v):
    X = rng.normal(size=(n, n))
    Hm = 0.5 * (X + X.T)
    w = np.linalg.eigvalsh(Hm)
    Hm = 2.0 * (Hm - w.mean() * np.eye(n)) / (w[-1] - w[0])
    bath = _drude(0.2, 1.0, 0.5, modes)
    noises = []
    for _ in range(baths):
        if dense_v:
            Y = rng.normal(size=(n, n))
            V = 0.5 * (Y + Y.T) / math.sqrt(2.0 * n)
        else:
            V = np.diag((rng.random(n) < 0.5).astype(np.float64))
        noises.append(_noise(V, bath))
    return {"N": n, "H": Hm.astype(np.complex128), "noises": noises, "max_depth": depth}


def _closure_model(rng, n, modes, depth):
    """Chain in units of the bath rate, as the closure is trained on."""
    J = rng.uniform(-1.0, 1.0, n - 1)
    e = rng.normal(0.0, 0.5, n)
    lam, T = rng.uniform(0.1, 1.0), rng.uniform(0.5, 2.0)
    bath = _drude(lam, 1.0, T, modes)
    noises = []
    for u in range(n):
        V = np.zeros((n, n))
        V[u, u] = 1.0
        noises.append(_noise(V, bath))
    Hm = np.diag(e) + np.diag(J, 1) + np.diag(J, -1)
    return {"N": n, "H": Hm.astype(np.complex128), "noises": noises, "max_depth": depth,
            "features": np.array([lam, T, *e, *J], np.float32)}


def _models(case, rng):
    """The case's systems (one, but for a sweep)."""
    f = case["family"]
    if f == "spin_boson":
        sx, sz = np.array([[0, 1], [1, 0.0]]), np.array([[1, 0], [0, -1.0]])
        Hm = 0.5 * rng.uniform(-1.0, 1.0) * sz + rng.uniform(0.5, 1.5) * sx
        bath = _drude(rng.uniform(0.3, 0.7), 1.0, rng.uniform(0.8, 1.2), case["modes"])
        return [{"N": 2, "H": Hm.astype(np.complex128), "noises": [_noise(sz, bath)],
                 "max_depth": case["depth"]}]
    if f in ("chain", "liou", "ado"):
        return [_chain_model(rng, case["sites"], case["modes"], case["depth"])]
    if f in ("dense", "dense_v"):
        return [_dense_model(rng, case["levels"], case["baths"], case["modes"], case["depth"],
                             f == "dense_v")]
    if f == "closure":
        return [_closure_model(rng, case["sites"], case["modes"], case["depth"])]
    # sweep: N, number of modes and depth follow the member's index (the same
    # total for every seed), the Hamiltonian, coupling and bath the seed
    out = []
    shape = np.random.default_rng(case["members"])
    for _ in range(case["members"]):
        n, modes = int(shape.choice([2, 4, 8])), int(shape.integers(2, 5))
        depth = int(shape.integers(4, 13))
        X = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
        signs = np.where(rng.random(n) < 0.5, 1.0, -1.0)
        signs[0], signs[-1] = 1.0, -1.0
        bath = _drude(rng.uniform(0.05, 2.0), rng.uniform(0.2, 1.5), rng.uniform(0.5, 1.0), modes)
        out.append({"N": n, "H": 0.5 * (X + X.conj().T), "noises": [_noise(np.diag(signs), bath)],
                    "max_depth": depth})
    return out


def _n_modes(m):
    return sum(len(z["phi_0"]) for z in m["noises"])


def _n_ado(m):
    return math.comb(_n_modes(m) + m["max_depth"], m["max_depth"])


def _state(m, rng, filled):
    """A random density matrix in ADO 0; `filled`: a state in mid-run, with the
    other ADOs populated as well."""
    n, a = m["N"], _n_ado(m)
    v = rng.normal(size=(n, n)) + 1j * rng.normal(size=(n, n))
    r = v @ v.conj().T
    rho = np.zeros((a, n, n), np.complex128)
    if filled:
        rho[...] = 0.05 * (rng.normal(size=rho.shape) + 1j * rng.normal(size=rho.shape)) / n
    rho[0] = r / np.trace(r).real
    return rho.reshape(-1)


def _network(case, rng, n_in, n_hid, n_out):
    """Parameters (heom_mlp's order) and scaling of a network, FP32."""
    def layer(o, i):
        b = math.sqrt(6.0 / (i + o))
        return [rng.uniform(-b, b, o * i), rng.normal(size=o) * 0.1]
    p = np.concatenate(layer(n_hid, n_in) + layer(n_hid, n_hid) + layer(n_out, n_hid))
    sc = [rng.normal(size=n_in) * 0.1, rng.uniform(0.5, 2.0, n_in), rng.normal(size=n_out) * 0.01,
          rng.uniform(0.05, 0.2, n_out)]
    return p.astype(np.float32), [s.astype(np.float32) for s in sc]


def _times(case):
    step = case["t_out"] if case.get("method") == "rkdp" else case["dt"] * case["steps"]
    return step * np.arange(case["outputs"] + 1)


def _kwargs(case):
    if case.get("method") == "rkdp":
        return {"dt": case["dt"], "rtol": case["rtol"], "atol": 1e-3 * case["rtol"]}
    return {"dt": case["dt"]}


def _inputs(case, seed):
    """Everything the seed decides, as host arrays."""
    rng = np.random.default_rng(int(seed))
    f = case["family"]
    if f == "grad":
        p, sc = _network(case, rng, case["inputs"], case["hidden"], case["targets"])
        X = rng.normal(size=(case["rows"], case["inputs"])).astype(np.float32)
        Y = (0.1 * rng.normal(size=(case["rows"], case["targets"]))).astype(np.float32)
        return {"params": p, "scaling": sc, "X": X, "Y": Y}
    ms = _models(case, rng)
    filled = case.get("method") != "rkdp"
    d = {"models": ms, "rho": [_state(m, rng, filled) for m in ms]}
    if f == "closure":
        m = ms[0]
        n2, k = m["N"] ** 2, _n_modes(m)
        d["dims"] = (2 * n2 + k + len(m["features"]), case["hidden"], 2 * n2)
        d["params"], d["scaling"] = _network(case, rng, *d["dims"])
    return d


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
def _host_ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def prepare(case, seed):
    d = _inputs(case, seed)
    f = case["family"]
    s = {"case": case}
    if f == "grad":
        net = C.Mlp(case["inputs"], case["hidden"], case["targets"])
        net.set_params(d["params"])
        net.set_scaling(*d["scaling"])
        s.update(net=net, X=torch.from_numpy(d["X"]).cuda(), Y=torch.from_numpy(d["Y"]).cuda(),
                 grad=np.zeros(net.n_params, np.float32), loss=ctypes.c_double())
        return s
    eng = H.hip(0)
    dtype = case.get("dtype", "complex128")
    form = {"liou": H.heom_liou, "ado": H.heom_ado}.get(f, H.heom_hilb)
    qs = [form(m["max_depth"], dtype=dtype).load(m, eng) for m in d["models"]]
    q = H.heom_batch(qs) if f == "sweep" else qs[0]
    rho = q.pack(d["rho"]) if f == "sweep" else d["rho"][0]
    s["qme"] = q
    if f == "dense_v":
        low = dtype == "complex64"
        s["rho"] = torch.from_numpy(rho.astype(np.complex64) if low else rho).cuda()
        s["drho"] = torch.empty_like(s["rho"])
        return s
    if f == "closure":
        net = C.Mlp(*d["dims"])
        net.set_params(d["params"])
        net.set_scaling(*d["scaling"])
        q.set_closure(net, d["models"][0]["features"])
        s["net"] = net
    method = H.rkdp() if case.get("method") == "rkdp" else H.rk4()
    s["solver"] = H.qme_solver(eng, q, method)
    s["t"], s["kw"] = np.ascontiguousarray(_times(case)), _kwargs(case)
    if case.get("entry"):
        s["rho"] = rho
    else:
        s["rho"] = torch.from_numpy(rho).cuda()
        n2 = q.rho_s_size() if f == "sweep" else q.n_level ** 2
        s["rho_s"] = np.zeros((s["t"].size, n2), np.complex128)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    case, f = s["case"], s["case"]["family"]
    L = _capi.load()
    if f == "grad":
        _capi.check(L.heom_mlp_loss_grad(s["net"]._h, s["X"].data_ptr(), s["Y"].data_ptr(),
                                         case["rows"], ctypes.byref(s["loss"]),
                                         _host_ptr(s["grad"])))
        return s["loss"].value, s["grad"].copy()
    if f == "dense_v":
        s["qme"].calc_diff_dev(s["drho"].data_ptr(), s["rho"].data_ptr(), 1.0, 0.0)
        return s["drho"]
    sv = s["solver"]
    sv.reset()  # every pass is a solve of its own: no step size from the last one
    if case.get("entry") == "solve":
        rho, seen = s["rho"].copy(), []
        n2 = s["qme"].n_level ** 2
        sv.solve(rho, s["t"], lambda t: seen.append(rho[:n2].copy()), s["kw"])
        return rho, np.stack(seen)
    if case.get("entry") == "solve_rho_s":
        rho, rho_s = sv.solve_rho_s(s["rho"], s["t"], s["kw"])
        return rho, rho_s.reshape(s["t"].size, -1)
    rho, kw = s["rho"].clone(), s["kw"]
    _capi.check(L.heom_solve_dev(sv._s, rho.data_ptr(), _host_ptr(s["t"]), s["t"].size, kw["dt"],
                                 kw.get("atol", 0.0), kw.get("rtol", 0.0),
                                 _host_ptr(s["rho_s"])))
    rho_s = s["rho_s"].copy()
    if case.get("dtype", "complex128") != "complex128" or f == "closure":
        # an FP32 operator (or network): the results are kept in the precision they have
        return rho.to(torch.complex64), rho_s.astype(np.complex64)
    return rho, rho_s


# ---------------------------------------------------------------------------
# what it cannot do without
# ---------------------------------------------------------------------------
def _evaluations(case):
    """Derivative evaluations of a pass (adaptive: about what the models take)."""
    if case["family"] == "dense_v":
        return 1
    if case.get("method") != "rkdp":
        return 4 * case["outputs"] * case["steps"]
    rate = {"spin_boson": 40.0, "chain": 0.6, "dense": 50.0}[case["family"]]
    tol = (1e-8 / case["rtol"]) ** 0.2
    return 7 * max(case["outputs"] * 2, int(case["outputs"] * case["t_out"] * rate * tol))


def work(case):
    """Per evaluation: the commutator with a real H (8 N^3 flops per ADO), the
    neighbour couplings (8 N^2 per link) and the stage combination; a state
    larger than one compute unit's LDS streams through memory in every stage
    (rk4: input, y and accumulator read, next input and accumulator written;
    Dormand-Prince: 40 blocks in seven stages), a smaller one once per solve."""
    if case["family"] == "grad":
        r, i, h, o = case["rows"], case["inputs"], case["hidden"], case["targets"]
        par = h * i + h * h + o * h
        return {"bytes": 4.0 * (r * (i + o) + 2 * par),
                "flops": 2.0 * r * (3 * h * h + 3 * o * h + 2 * h * i)}
    ms = _models(case, np.random.default_rng(0))
    ev = _evaluations(case)
    wide = case.get("dtype", "complex128") == "complex128"
    nbytes = flops = 0.0
    for m in ms:
        n, k, a = m["N"], _n_modes(m), _n_ado(m)
        links = 2.0 * k * math.comb(k + m["max_depth"] - 1, k) if m["max_depth"] else 0.0
        per = 8.0 * n ** 3 * a + 8.0 * n * n * links + 12.0 * n * n * a
        if case["family"] == "dense_v":
            per += len(m["noises"]) * 16.0 * n ** 3 * a
        if case["family"] == "closure":
            last = math.comb(k + m["max_depth"] - 1, m["max_depth"])
            h, i, o = case["hidden"], 2 * n * n + k + 2 + 2 * n - 1, 2 * n * n
            per += 2.0 * last * (h * i + h * h + o * h)
        flops += ev * per
        state = a * n * n * 16.0
        if case["family"] == "dense_v":
            nbytes += 2 * state * (1.0 if wide else 0.5)
        elif state * 4 < 160 * 1024:
            nbytes += 2 * state
        else:
            blocks = 40.0 / 7.0 if case.get("method") == "rkdp" else 5.0
            nbytes += ev * blocks * state * (1.0 if wide else 0.7)
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _hierarchy(k, depth):
    """Indices in breadth-first order and the +-1 neighbours (the count where
    there is none)."""
    order, queue = [], [((0,) * k, 0, 0)]
    for idx, last, d in queue:
        order.append(idx)
        if d < depth:
            for j in range(last, k):
                queue.append((idx[:j] + (idx[j] + 1,) + idx[j + 1:], j, d + 1))
    book = {x: i for i, x in enumerate(order)}
    a = len(order)
    p1, m1 = np.full((k, a), a), np.full((k, a), a)
    for i, x in enumerate(order):
        for j in range(k):
            if x[j]:
                b = book[x[:j] + (x[j] - 1,) + x[j + 1:]]
                m1[j, i] = b
                p1[j, b] = i
    return np.array(order, np.int64).reshape(a, k), p1, m1


class _Operator:
    """D of the hierarchical equations for systems of one size N, their ADOs
    one after another."""

    def __init__(self, models, device):
        n = models[0]["N"]
        self.N, self.n_noise = n, len(models[0]["noises"])
        slots = max(_n_modes(m) for m in models)
        base, hs, tabs = 0, [], {}
        for m in models:
            k, depth = _n_modes(m), m["max_depth"]
            if (k, depth) not in tabs:
                tabs[k, depth] = _hierarchy(k, depth)
            hs.append((base,) + tabs[k, depth])
            base += len(hs[-1][1])
        A = self.A = base
        gam = np.zeros(A, np.complex128)
        p1, m1 = np.full((slots, A), A), np.full((slots, A), A)
        cp, cf, cs = (np.zeros((slots, A), np.complex128) for _ in range(3))
        one = len(models) == 1
        Hm = np.zeros((1 if one else A, n, n), np.complex128)
        V = np.zeros((self.n_noise, 1 if one else A, n, n), np.complex128)
        dl = np.zeros((self.n_noise, 1 if one else A), np.complex128)
        self.noise_of = []
        for m, (b, idx, q1, r1) in zip(models, hs):
            a = len(idx)
            at = slice(0, 1) if one else slice(b, b + a)
            Hm[at] = m["H"]
            j = 0
            self.noise_of = []
            for u, z in enumerate(m["noises"]):
                V[u, at], dl[u, at] = z["V"], z["s_delta"]
                sc, ac = z["S"] @ z["phi_0"], z["A"] @ z["phi_0"]
                for i in range(len(sc)):
                    occ = idx[:, j]
                    gam[b:b + a] += occ * z["gamma"][i, i]
                    p1[j, b:b + a] = np.where(q1[j] == a, A, q1[j] + b)
                    m1[j, b:b + a] = np.where(r1[j] == a, A, r1[j] + b)
                    cp[j, b:b + a] = z["sigma"][i]
                    cf[j, b:b + a] = occ * sc[i]
                    cs[j, b:b + a] = -occ * ac[i]
                    self.noise_of.append(u)
                    j += 1
        self.noise_of += [0] * (slots - len(self.noise_of))
        t = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(device)  # noqa: E731
        col = lambda x: t(x).reshape(*x.shape, 1, 1)                        # noqa: E731
        self.H, self.V, self.dl, self.gam = t(Hm), t(V), col(dl), col(gam)
        self.p1, self.m1, self.cp, self.cf, self.cs = t(p1), t(m1), col(cp), col(cf), col(cs)
        off = V.copy()
        off[..., np.arange(n), np.arange(n)] = 0
        self.diag = not off.any()
        self.last = (hs[0][1].sum(1) == models[0]["max_depth"]).nonzero()[0]
        self.index = hs[0][1]
        self.device = device
        self.extra = None

    def _both(self, u, X, Y):
        """V X - X V and V Y + Y V."""
        V = self.V[u]
        if self.diag:
            v = torch.diagonal(V, dim1=-2, dim2=-1)
            vi, vj = v[:, :, None], v[:, None, :]
            return (vi - vj) * X, (vi + vj) * Y
        return V @ X - X @ V, V @ Y + Y @ V

    def __call__(self, X):
        D = 1j * (self.H @ X - X @ self.H) + self.gam * X
        Xp = torch.cat([X, torch.zeros_like(X[:1])])
        for u in range(self.n_noise):
            phi, psi = torch.zeros_like(X), torch.zeros_like(X)
            for j, v in enumerate(self.noise_of):
                if v != u:
                    continue
                up, dn = Xp[self.p1[j]], Xp[self.m1[j]]
                phi += self.cp[j] * up + self.cf[j] * dn
                psi += self.cs[j] * dn
            a, b = self._both(u, phi, psi)
            c, _ = self._both(u, X, X)
            c, _ = self._both(u, c, c)
            D += 1j * a + b + self.dl[u] * c
        if self.extra is not None:
            self.extra(X, D)
        return D


_A = [[], [1 / 5], [3 / 40, 9 / 40], [44 / 45, -56 / 15, 32 / 9],
      [19372 / 6561, -25360 / 2187, 64448 / 6561, -212 / 729],
      [9017 / 3168, -355 / 33, 46732 / 5247, 49 / 176, -5103 / 18656],
      [35 / 384, 0.0, 500 / 1113, 125 / 192, -2187 / 6784, 11 / 84]]
_E = [-71 / 57600, 0.0, 71 / 16695, -71 / 1920, 17253 / 339200, -22 / 525, 1 / 40]


def _fixed(f, y, t, dt):
    """Classical RK4 over the output times; the last step of an interval ends on it."""
    eps, out = np.finfo(np.float64).eps, [y]
    for t0, t1 in zip(t[:-1], t[1:]):
        at, last = t0, False
        while not last:
            h = dt
            if at + h - t1 > -eps:
                h, last = t1 - at, True
            k1 = -h * f(y)
            k2 = -h * f(y + 0.5 * k1)
            k3 = -h * f(y + 0.5 * k2)
            k4 = -h * f(y + k3)
            y = y + (k1 + 2 * k2 + 2 * k3 + k4) / 6
            at += h
        out.append(y)
    return y, out


def _adaptive(f, y, t, dt, atol, rtol):
    """Dormand-Prince 5(4), the step factor 0.9 err^(-1/5) within [0.2, 10]."""
    out = [y]
    for t0, t1 in zip(t[:-1], t[1:]):
        at = t0
        h = min(dt, t1 - at)
        while True:
            k = []
            for i in range(7):
                s = y
                for a, kk in zip(_A[i], k):
                    if a:
                        s = s + a * kk
                k.append(-h * f(s))
            e = sum(c * kk for c, kk in zip(_E, k) if c)
            w = e.abs() / (atol + rtol * torch.maximum(s.abs(), y.abs()))
            err = float(w.square().mean().sqrt())
            fac = err ** -0.2 if err > 0 else math.inf
            if err < 1.0:
                at += h
                y = s
                h *= 0.9 * min(fac, 10.0)
                if at >= t1:
                    break
            else:
                h = max(h * 0.9 * max(fac, 0.2), 1e-16)
            h = min(h, t1 - at)
        dt = h
        out.append(y)
    return y, out


def _unpack(p, i, h, o):
    p, parts, at = p.double(), [], 0
    for shape in ((h, i), (h,), (h, h), (h,), (o, h), (o,)):
        n = math.prod(shape)
        parts.append(p[at:at + n].reshape(shape))
        at += n
    return parts


def _exact_grad(case, d):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda x: torch.from_numpy(x).to(dev)  # noqa: E731
    p = t(d["params"]).double().requires_grad_(True)
    W1, b1, W2, b2, W3, b3 = _unpack(p, case["inputs"], case["hidden"], case["targets"])
    xm, xs, ym, ys = (t(v).double() for v in d["scaling"])
    x, y = (t(d["X"]).double() - xm) / xs, (t(d["Y"]).double() - ym) / ys
    out = torch.tanh(torch.tanh(x @ W1.T + b1) @ W2.T + b2) @ W3.T + b3
    loss = (out - y).square().mean()
    g, = torch.autograd.grad(loss, p)
    return float(loss.detach()), g.detach().cpu().numpy()


def exact(case, seed):
    d = _inputs(case, seed)
    f = case["family"]
    if f == "grad":
        return _exact_grad(case, d)
    ms = d["models"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    sizes = sorted({m["N"] for m in ms})
    whole, small = [None] * len(ms), [None] * len(ms)
    for n in sizes:
        at = [i for i, m in enumerate(ms) if m["N"] == n]
        op = _Operator([ms[i] for i in at], dev)
        y = torch.from_numpy(np.concatenate([d["rho"][i] for i in at])).to(dev)
        if f == "dense_v" and case.get("dtype") == "complex64":
            y = y.to(torch.complex64).to(torch.complex128)
        y = y.reshape(-1, n, n)
        if f == "dense_v":
            return -op(y).reshape(-1)
        if f == "closure":
            W1, b1, W2, b2, W3, b3 = _unpack(torch.from_numpy(d["params"]).to(dev), *d["dims"])
            xm, xs, ym, ys = (torch.from_numpy(v).to(dev).double() for v in d["scaling"])
            last = torch.from_numpy(op.last).to(dev)
            fixed = np.concatenate([op.index[op.last], np.tile(
                ms[0]["features"].astype(np.float64), (len(op.last), 1))], 1)
            fixed = torch.from_numpy(fixed).to(dev)

            def add(X, D):
                x = X[last].reshape(len(last), -1)
                x = (torch.cat([x.real, x.imag, fixed], 1) - xm) / xs
                p = torch.tanh(torch.tanh(x @ W1.T + b1) @ W2.T + b2) @ W3.T + b3
                p = p * ys + ym
                D[last] += torch.complex(p[:, :n * n], p[:, n * n:]).reshape(-1, n, n)
            op.extra = add
        kw = _kwargs(case)
        if case.get("method") == "rkdp":
            y, seen = _adaptive(op, y, _times(case), kw["dt"], kw["atol"], kw["rtol"])
        else:
            y, seen = _fixed(op, y, _times(case), kw["dt"])
        b = 0
        for i in at:
            a = _n_ado(ms[i])
            whole[i] = y[b:b + a].reshape(-1)
            small[i] = torch.stack([s[b].reshape(-1) for s in seen])
            b += a
    rho, rho_s = torch.cat(whole), torch.cat(small, 1)
    return (rho if not case.get("entry") else rho.cpu().numpy()), rho_s.cpu().numpy()
