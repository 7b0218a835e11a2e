"""Benchmark: HEOM propagation of the 7-site exciton chain on one MI355X.

Workload (one "step" = one full propagation, the time-to-rho_S(t) job):
  7-site chain, N = 7, per-site Drude bath (1 Drude + 2 Pade modes) -> K = 21,
  depth L = 4 -> 12650 ADOs (main_size 619850 complex128), Dormand-Prince
  rtol = 1e-8, atol = 1e-11, t = 0 .. 1000 fs, rho_S recorded every 10 fs,
  plain FP64 (complex128) Hilbert form.  Inputs are synthetic (seeded).
The state is resident in HBM when the timed region starts.

Metric: ADO-stage updates/s = n_hrchy * (RHS evaluations performed) / s.  A
Dormand-Prince attempt has seven stages; the first is the last one of the attempt
before, so six evaluations are performed (evaluations()).
Also reported: the roofline of the dominant kernel (the fused Hilbert-form
stage pass; the bytes the pass itself must move per launch / average launch
duration measured with HIP events on the library stream, over the six operator
passes of an attempt) and the CPU oracle timed on the host cores on a bounded
sample of the same workload.  Beside it the same attempt, step pass included,
against the bytes of the reference's step (alg_bytes_per_ado_stage, seven
evaluations without fusion of the error sum).

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W]
"""
import argparse
import ctypes
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
GRAPHS = True  # resident launches and graph replay (--no-graphs: every stage launched)


def alg_bytes_per_ado_stage(n_level, n_dim, method, sc=16):
    """Algorithmic HBM bytes of one ADO-stage of the reference's stepping:
    m N^2-blocks of sc bytes (sc = 16 complex128, 8 complex64), two int32
    neighbour indices per mode and Gamma_n.  Dormand-Prince without FSAL
    (rkdp.h:108-146): stage i of 1..6 reads y_i, y, k_1..k_{i-1} and writes k_i
    and y_{i+1} (i + 3 blocks), stage 7 with the error norm moves 8: m = 47/7.
    Fused RK4 (rk4.h:40-65): y_s, y, acc read, y_{s+1}, acc written: m = 5.
    Neighbour ADOs count once (another ADO's compulsory read)."""
    m = 47.0 / 7.0 if method == "rkdp" else 5.0
    return m * n_level * n_level * sc + 8.0 * n_dim + 8.0


def evaluations(st, solves=1, projected=False):
    """Operator evaluations of `solves` Dormand-Prince solves: six per attempt and one
    at the start of each, or seven per attempt where rho_0 is projected (the stored
    derivative is stale then).  stats()["n_rhs"] counts the scheme's stages, seven per
    attempt."""
    return 7 * st["n_attempts"] if projected else 6 * st["n_attempts"] + solves


def mk_solver(H, eng, q, method):
    sv = H.qme_solver(eng, q, method)
    sv.set_graphs(GRAPHS)
    return sv
TRAFFIC_JSON = os.path.join(ROOT, "profiles", "hilb_fast_kernel_7site_traffic.json")


def _pmc_rows(path, counter):
    """(kernel name, grid size, value) of every dispatch in a rocprofv3 counter
    run: its SQLite results file (*_results.db) or counter_collection.csv."""
    if path.endswith(".db"):
        import sqlite3
        con = sqlite3.connect(path)
        q = ("select kernel_name, grid_size, value from counters_collection "
             "where counter_name = ?")
        return [(k, int(g), float(v)) for k, g, v in con.execute(q, (counter,))]
    import csv
    return [(r["Kernel_Name"], int(r["Grid_Size"]), float(r["Counter_Value"]))
            for r in csv.DictReader(open(path)) if r["Counter_Name"] == counter]


def summarize_pmc(fetch_path, write_path, state_bytes, kernel="hilb_fast_kernel<7, double"):
    """HBM bytes per dispatch of the stage kernel from two rocprofv3 --pmc runs
    (FETCH_SIZE, WRITE_SIZE; KiB per dispatch).  Each counter is scaled by what
    it reads for the largest rocclr copy in the same run, a device-to-device
    copy of one state buffer (state_bytes read, state_bytes written).  Dispatches
    that leave at once (a finished Dormand-Prince interval) are left out: they
    move less than 1% of a state buffer."""
    import statistics

    def load(path, counter):
        rows = _pmc_rows(path, counter)
        copies = [r for r in rows if "copyBuffer" in r[0]]
        big = max(r[1] for r in copies)
        cal = statistics.median(r[2] for r in copies if r[1] == big)
        stage = [r[2] for r in rows if kernel in r[0]]
        floor = 0.01 * state_bytes / 1024.0
        live = [v for v in stage if v > floor]
        return statistics.mean(live), cal, len(live), len(stage) - len(live)

    f, fcal, n1, e1 = load(fetch_path, "FETCH_SIZE")
    w, wcal, n2, e2 = load(write_path, "WRITE_SIZE")
    fs, ws = state_bytes / (fcal * 1024.0), state_bytes / (wcal * 1024.0)
    return {"kernel": kernel, "fetch_bytes": f * 1024.0 * fs, "write_bytes": w * 1024.0 * ws,
            "traffic": f * 1024.0 * fs + w * 1024.0 * ws,
            "fetch_scale": fs, "write_scale": ws, "dispatches": [n1, n2],
            "early_exit_dispatches_left_out": [e1, e2],
            "fetch_kib_raw": f, "write_kib_raw": w}


def summarize_trace(path, top=12, live_us=5.0):
    """Markdown table of a rocprofv3 --kernel-trace run (its *_results.db):
    per kernel the dispatches, total time, mean, and the mean over dispatches of
    at least live_us (the stage passes of a finished Dormand-Prince interval
    leave at once and take about 3 us)."""
    import sqlite3
    import statistics
    con = sqlite3.connect(path)
    rows = list(con.execute("select name, duration from kernels"))
    by = {}
    for name, dur in rows:
        by.setdefault(name, []).append(dur / 1e3)  # us
    total = sum(sum(v) for v in by.values())
    out = ["| kernel | dispatches | total ms | %% | mean us | dispatches >= %g us | their mean us |"
           % live_us, "|---|---|---|---|---|---|---|"]
    for name, v in sorted(by.items(), key=lambda kv: -sum(kv[1]))[:top]:
        live = [x for x in v if x >= live_us]
        short = name.replace("void ", "").replace("hamd::(anonymous namespace)::", "")
        short = short.replace("(hamd::Epi)", "").replace("hamd::", "").split("(")[0]
        out.append("| `%s` | %d | %.2f | %.1f | %.2f | %d | %s |" % (
            short, len(v), sum(v) / 1e3, 100.0 * sum(v) / total, statistics.mean(v), len(live),
            "%.2f" % statistics.mean(live) if live else "-"))
    return "\n".join(out)


def _host_cpu():
    """(cores used, nproc, model name) of the host: the threads are the cores this
    process may run on, bounded by OMP_NUM_THREADS when the machine sets it (the
    CPU share the host gives this job)."""
    try:
        cores = len(os.sched_getaffinity(0))
    except AttributeError:
        cores = os.cpu_count() or 1
    nproc = cores
    env = os.environ.get("OMP_NUM_THREADS")
    if env and env.isdigit() and int(env) > 0:
        cores = min(cores, int(env))
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return max(1, cores), nproc, model


def cpu_baseline(m, attempts=6, runs=5):
    """Oracle (FP64 CPU restatement) on a bounded sample of the same workload:
    `attempts` Dormand-Prince attempts from rho(0), OpenMP over ADOs on the host
    cores; one warm-up run, then `runs` timed runs (median, min, max)."""
    from oracle import oracle as O
    import statistics
    cores, nproc, model = _host_cpu()
    o = O.Oracle(O.HILB, m["N"], m["max_depth"], n_threads=cores).load(m)

    def one():
        rho = m["rho0"].copy()
        t, dt, n_rhs, done = 0.0, m["dt"], 0, 0
        t0 = time.perf_counter()
        while done < attempts:
            rho, t, dt, st, rc = o.rkdp_step(rho, t, m["t_list"][-1], dt, m["atol"], m["rtol"])
            n_rhs += st.n_rhs
            done += st.n_accepted + st.n_rejected
        return o.n_hrchy * n_rhs / (time.perf_counter() - t0), n_rhs

    one()  # warm-up
    vals = [one() for _ in range(runs)]
    rates = [v for v, _ in vals]
    return {
        "value": statistics.median(rates), "unit": "ADO-stage updates/s", "cores": cores,
        "kind": "port", "min": min(rates), "max": max(rates), "runs": runs,
        "nproc": nproc, "cpu_model": model,
        "sample": "%d Dormand-Prince attempts (%d RHS evaluations) of the same 12650-ADO "
                  "workload from rho(0), OpenMP over ADOs on %d threads; 1 warm-up + %d "
                  "timed runs, median" % (attempts, vals[0][1], cores, runs),
    }


def stream_copy_roof(L):
    """The project's grid-stride copy kernel: HBM-sized (2 GiB) and
    Infinity-Cache-resident (40 MiB) buffers, best grid of three."""
    from libheom_amd import _capi
    out = {}
    for name, nb in (("hbm_2GiB", 2 << 30), ("mall_40MiB", 40 << 20)):
        best = 0.0
        for grid in (1024, 4096, 16384):
            g = ctypes.c_double()
            _capi.check(L.heom_stream_copy(nb, grid, 10, ctypes.byref(g)))
            best = max(best, g.value)
        out[name] = best
    out["unit"] = "GB/s (read + write)"
    out["spec_hbm"] = HBM_PEAK_GBS
    out["hbm_frac_of_spec"] = out["hbm_2GiB"] / HBM_PEAK_GBS
    return out


GOLDEN = os.path.join(ROOT, "tests", "golden")


def golden_rho_s(name):
    """rho_S(t) of the oracle's committed run of a workload (None if absent)."""
    path = os.path.join(GOLDEN, name)
    if not os.path.exists(path):
        return None
    return np.load(path)["rho_s"]


def bench_sweep(H, L, steps, warmup, reps):
    """512-instance parameter sweep (N in {2,4,8}, K 2..4, L 4..12), RK4
    dt=0.005 x 4000 steps, advanced as one batch: complex64 operator with FP64
    stage combination (the sweep's stated precision), the FP64 batch beside it
    for the error, and a sample of members run one at a time for comparison."""
    from libheom_amd import _capi, configs
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    ms = configs.batched_sweep()
    t_list = np.ascontiguousarray(ms[0]["t_list"])
    dt = ms[0]["dt"]
    eng = H.hip(0)
    res = {}
    for dtype in ("complex64", "complex128"):
        qs = [H.heom_hilb(m["max_depth"], dtype=dtype).load(m, eng) for m in ms]
        unit = sum(q.n_hrchy * alg_bytes_per_ado_stage(q.n_level, q.n_dim, "rk4",
                                                       8 if dtype == "complex64" else 16)
                   for q in qs)
        b = H.heom_batch(qs)
        sv = mk_solver(H, eng, b, H.rk4())
        rho0 = b.pack([m["rho0"] for m in ms])
        nb = rho0.nbytes
        d = ctypes.c_void_p()
        _capi.check(L.heom_dev_alloc(ctypes.byref(d), nb))
        rs = np.zeros((t_list.size, b.rho_s_size()), np.complex128)

        def run():
            _capi.check(L.heom_memcpy_h2d(d, p(rho0), nb))
            _capi.check(L.heom_device_sync())
            t0 = time.perf_counter()
            _capi.check(L.heom_solve_dev(sv._s, d, p(t_list), t_list.size, dt, 0.0, 0.0, p(rs)))
            _capi.check(L.heom_device_sync())
            return time.perf_counter() - t0

        for _ in range(warmup):
            run()
        sv.reset()
        el = sum(run() for _ in range(steps))
        st = sv.stats()
        ns = ctypes.c_int()
        sms, sby = np.zeros(8), np.zeros(8)
        _capi.check(L.heom_solver_time_stages(sv._s, reps, p(sms), ctypes.byref(ns)))
        _capi.check(L.heom_solver_stage_bytes(sv._s, p(sby), ctypes.byref(ns)))
        n = ns.value
        gbs = unit / (float(sms[:n].mean()) * 1e-3) / 1e9
        gbs_kernel = float(sby[:n].mean()) / (float(sms[:n].mean()) * 1e-3) / 1e9
        final = np.zeros_like(rho0)
        _capi.check(L.heom_memcpy_d2h(p(final), d, nb))
        L.heom_dev_free(d)
        chosen, tried = b.tuning()
        res[dtype] = {"value": st["ado_stage_updates"] / el, "ms_per_step": 1e3 * el / steps,
                      "autotune": dict(chosen, tried_us_per_pass={
                          "ipw%d_wpb%d_grid%d" % (k, w, g): round(u, 1) for k, w, g, u in tried}),
                      "stage_ms": float(sms[:n].mean()), "stage_bytes": float(sby[:n].mean()),
                      "hbm_frac": gbs / HBM_PEAK_GBS, "alg_bytes_per_stage": unit,
                      "hbm_frac_kernel_bytes": gbs_kernel / HBM_PEAK_GBS, "rs": b.split_rho_s(rs),
                      "final": b.unpack(final),
                      "n_hrchy": b.n_hrchy, "main_size": b.main_size()}
    # members whose FP64 rho_S stays a bounded density matrix (|rho_ij| <= 1);
    # the others grow without bound (RK4 at dt=0.005 is outside its stability
    # region for their largest Pade frequency x depth) and carry no error figure
    # stable members: the whole FP64 hierarchy stays below 1e4 as well (members whose
    # deep ADOs grow amplify the FP32 rounding even while rho_S stays bounded)
    worst, n_div, worst_st, n_st = 0.0, 0, 0.0, 0
    for a, r, full in zip(res["complex64"]["rs"], res["complex128"]["rs"],
                          res["complex128"]["final"]):
        if not np.isfinite(r).all() or np.abs(r).max() > 1.0 + 1e-6:
            n_div += 1
            continue
        e = float(np.abs(a - r).max())
        worst = max(worst, e)
        if np.isfinite(full).all() and np.abs(full).max() <= 1e4:
            n_st += 1
            worst_st = max(worst_st, e)
    # members one at a time (FP64, same solver): a sample, scaled to 512 by ADO count
    sample = ms[::64]
    t_one, ado_one = 0.0, 0
    for m in sample:
        q = H.heom_hilb(m["max_depth"]).load(m, eng)
        sv = mk_solver(H, eng, q, H.rk4())
        t0 = time.perf_counter()
        sv.solve_rho_s(m["rho0"], t_list, {"dt": dt})
        t_one += time.perf_counter() - t0
        ado_one += q.n_hrchy
    one_ms = 1e3 * t_one * res["complex128"]["n_hrchy"] / ado_one
    f32, f64 = res["complex64"], res["complex128"]
    return {
        "workload": "512 independent heom_hilb instances (N in {2,4,8}, 1 Drude + 1-3 Pade, "
                    "L 4..12), RK4 dt=0.005 x 4000 steps, rho_S every 100 steps, one batch",
        "n_hrchy_total": f64["n_hrchy"], "main_size": f64["main_size"],
        "dtype": "f32 operator / f64 combination", "value": f32["value"],
        "ms_per_step": f32["ms_per_step"], "stage_ms": f32["stage_ms"],
        "hbm_frac": f32["hbm_frac"], "hbm_frac_kernel_bytes": f32["hbm_frac_kernel_bytes"],
        "alg_bytes_per_stage": f32["alg_bytes_per_stage"], "autotune": f32["autotune"],
        "fp64": {"value": f64["value"], "ms_per_step": f64["ms_per_step"],
                 "stage_ms": f64["stage_ms"], "hbm_frac": f64["hbm_frac"],
                 "hbm_frac_kernel_bytes": f64["hbm_frac_kernel_bytes"],
                 "alg_bytes_per_stage": f64["alg_bytes_per_stage"],
                 "autotune": f64["autotune"]},
        "fp32_batch_speedup_vs_fp64_batch": f64["ms_per_step"] / f32["ms_per_step"],
        "rho_s_max_abs_err_vs_fp64_bounded_members": worst,
        "bounded_members": len(ms) - n_div,
        "members_unbounded_under_rk4": n_div,
        "stable_members": n_st,
        "rho_s_max_abs_err_vs_fp64_stable_members": worst_st,
        "note": "bounded: the FP64 rho_S stays a density matrix; stable: the whole FP64 "
                "hierarchy stays below 1e4 as well",
        "side_note_one_at_a_time": {
            "fp64_one_at_a_time_est_ms": one_ms,
            "fp64_batch_speedup_vs_one_at_a_time_fp64": one_ms / f64["ms_per_step"]},
    }


def bench_spin_boson(H):
    """The CPU-runnable reference case: spin-boson N=2, 2 modes, depth 10 (66
    ADOs), RK4 dt=0.01 x 2000 steps, rho_S every 10 steps.  Latency-bound (the
    whole state is 4 KB): reported as time-to-solution in the default mode (the
    resident integrator: one launch per output interval, state in LDS) and with
    every stage kernel launched one by one."""
    from libheom_amd import configs
    m = configs.spin_boson()
    eng = H.hip(0)
    q = H.heom_hilb(m["max_depth"]).load(m, eng)
    res = {}
    for graphs in (True, False):
        if graphs and not GRAPHS:
            continue
        sv = H.qme_solver(eng, q, H.rk4())
        sv.set_graphs(graphs)
        sv.solve_rho_s(m["rho0"], m["t_list"][:3], {"dt": m["dt"]})  # warm-up
        t0 = time.perf_counter()
        sv.solve_rho_s(m["rho0"], m["t_list"], {"dt": m["dt"]})
        res[graphs] = time.perf_counter() - t0
        st = sv.stats()
    return {"workload": "spin-boson N=2, 1 Drude + 1 Pade mode, depth 10 (66 ADOs), RK4 "
                        "dt=0.01 x 2000 steps, rho_S every 10 steps",
            "time_to_rho_s_ms_resident": 1e3 * res[True] if True in res else None,
            "time_to_rho_s_ms_direct_launches": 1e3 * res[False],
            "us_per_stage": 1e6 * min(res.values()) / 8000,
            "value": q.n_hrchy * 8000 / min(res.values())}


def bench_dense64(H, L, reps):
    """Large-N config: N=64 GOE Hamiltonian, 4 projector baths x (1 Drude + 3
    Pade) = 16 modes, depth 3 (969 ADOs of 64x64), Dormand-Prince rtol=1e-6 to
    t=20, FP64 and complex64 (FP32 operator, FP64 combination)."""
    from libheom_amd import _capi, configs
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    m = configs.dense64()
    eng = H.hip(0)
    t_list = np.ascontiguousarray(m["t_list"])
    kw = {"dt": m["dt"], "atol": m["atol"], "rtol": m["rtol"]}
    res = {}
    for dtype in ("complex128", "complex64", "complex64_bf16x3", "valu"):
        # "valu": FP64 on the vector-ALU kernel (matrix_cores off), for comparison
        q = H.heom_hilb(m["max_depth"], dtype="complex128" if dtype == "valu" else dtype,
                        matrix_cores=dtype != "valu").load(m, eng)
        sv = mk_solver(H, eng, q, H.rkdp())
        sv.solve_rho_s(m["rho0"], t_list[:2], kw)  # warm-up
        sv.reset()
        t_run = t_list if dtype != "valu" else t_list[:3]  # stage timing only
        t0 = time.perf_counter()
        _, rs = sv.solve_rho_s(m["rho0"], t_run, kw)
        el = time.perf_counter() - t0
        st = sv.stats()
        ns = ctypes.c_int()
        sms, sby = np.zeros(8), np.zeros(8)
        _capi.check(L.heom_solver_time_stages(sv._s, reps, p(sms), ctypes.byref(ns)))
        _capi.check(L.heom_solver_stage_bytes(sv._s, p(sby), ctypes.byref(ns)))
        n = ns.value
        stage_ms = float(sms[:n].mean())
        # real flops per ADO-stage of the commutator (two complex N^3 products; H real
        # symmetric here, so 4 real N^3 GEMMs) -- the MFMA-relevant part
        flops = q.n_hrchy * 4 * 2 * 64 ** 3
        unit = q.n_hrchy * alg_bytes_per_ado_stage(
            q.n_level, q.n_dim, "rkdp", 16 if dtype in ("complex128", "valu") else 8)
        evals = evaluations(st)
        res[dtype] = {"value": q.n_hrchy * evals / el, "time_to_rho_s_ms": 1e3 * el,
                      "stage_ms": stage_ms,
                      "hbm_frac": unit / (stage_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
                      "alg_bytes_per_stage": unit,
                      "hbm_frac_kernel_bytes": float(sby[:n].mean()) / (stage_ms * 1e-3)
                      / 1e9 / HBM_PEAK_GBS,
                      "commutator_tflops": flops / (stage_ms * 1e-3) / 1e12,
                      "rhs_evals": evals, "rs": rs}
    f64 = res["complex128"]

    def variant(r):
        return dict({k: v for k, v in r.items() if k != "rs"},
                    rho_s_max_abs_err_vs_fp64=float(np.abs(r["rs"] - f64["rs"]).max()),
                    speedup_time_to_rho_s=f64["time_to_rho_s_ms"] / r["time_to_rho_s_ms"])

    # the same hierarchy with dense V: every bath couples through a random real
    # symmetric V (unit spectral width); per ADO-stage 36 real 64^3 products on the
    # matrix cores (4 for i[H, rho], 8 per bath for [V, rho], V X and Y V)
    md = configs.dense64()
    rng = np.random.default_rng(65)
    for z in md["noises"]:
        X = rng.normal(size=(64, 64))
        Vs = 0.5 * (X + X.T)
        w = np.linalg.eigvalsh(Vs)
        z["V"] = (Vs / (w[-1] - w[0])).astype(np.complex128)
    dense_v = {}
    for dtype in ("complex128", "complex64"):
        q = H.heom_hilb(md["max_depth"], dtype=dtype).load(md, eng)
        sv = mk_solver(H, eng, q, H.rkdp())
        sv.solve_rho_s(md["rho0"], t_list[:2], kw)  # builds the stages
        st_ms, st_b = _stage_stats(L, sv, reps)
        fl = q.n_hrchy * 36 * 2 * 64 ** 3
        dense_v[dtype] = {"stage_ms": st_ms, "hbm_frac": st_b / (st_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
                          "mfma_tflops": fl / (st_ms * 1e-3) / 1e12}
    return {
        "dense_v": dict(dense_v, workload="N=64, 969 ADOs, 4 baths with dense real symmetric V, "
                                          "one Dormand-Prince stage pass (hilb_mfma_dense_kernel)"),
        "workload": "N=64 GOE H, 4 diagonal-projector baths x (1 Drude + 3 Pade), depth 3, "
                    "969 ADOs, Dormand-Prince rtol=1e-6 atol=1e-9, t=0..20",
        "kernel": "hilb_mfma_kernel<64> (f64 / f32 16x16x4 or bf16 16x16x32 MFMA commutator, "
                  "fused Dormand-Prince stage)",
        "fp64": {k: v for k, v in f64.items() if k != "rs"},
        "complex64": variant(res["complex64"]),
        "complex64_bf16x3": variant(res["complex64_bf16x3"]),
        "fp64_vector_alu_stage_ms": res["valu"]["stage_ms"],
    }


def _stage_stats(L, sv, reps):
    """Mean per-stage device time (ms, HIP events) and algorithmic bytes of a solver."""
    from libheom_amd import _capi
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    ns = ctypes.c_int()
    sms, sby = np.zeros(8), np.zeros(8)
    _capi.check(L.heom_solver_time_stages(sv._s, reps, p(sms), ctypes.byref(ns)))
    _capi.check(L.heom_solver_stage_bytes(sv._s, p(sby), ctypes.byref(ns)))
    n = ns.value
    return float(sms[:n].mean()), float(sby[:n].mean())


def bench_lsrk4(H, L, reps):
    """lsrk4 against rk4 on the 7-site chain (12650 ADOs): the low-storage scheme
    keeps two state buffers plus the accumulator, so each stage pass moves four
    state blocks instead of five."""
    from libheom_amd import configs
    m = configs.exciton_chain7(t_final=10.0)
    eng = H.hip(0)
    q = H.heom_hilb(m["max_depth"]).load(m, eng)
    out = {"workload": "7-site chain, 12650 ADOs, heom_hilb complex128: one stage pass of "
                       "each fixed-step solver (dt=0.01 fs)"}
    for name, cls in (("rk4", H.rk4), ("lsrk4", H.lsrk4)):
        sv = mk_solver(H, eng, q, cls())
        sv.solve_rho_s(m["rho0"], m["t_list"][:2], {"dt": 0.01})  # builds the stages
        st_ms, st_b = _stage_stats(L, sv, reps)
        out[name] = {"stage_us": 1e3 * st_ms, "bytes_per_stage": st_b,
                     "hbm_frac": st_b / (st_ms * 1e-3) / 1e9 / HBM_PEAK_GBS}
    out["lsrk4_stage_speedup"] = out["rk4"]["stage_us"] / out["lsrk4"]["stage_us"]
    return out


def bench_redfield(H, L, reps, cpu=True):
    """Redfield QMEs (redfield_hilb / redfield_liou).  The states are one density
    matrix, so the small cases are launch-latency bound and are reported as
    time-to-solution next to the CPU oracle on the same job; the N=64 case runs
    the two-pass Hilbert kernels."""
    from libheom_amd import configs
    from oracle import oracle as O
    eng = H.hip(0)
    out = {}

    def timed(q, solver, m, t_list, kw, okind, oracle_solver):
        sv = mk_solver(H, eng, q, solver)
        sv.solve_rho_s(m["rho0"], t_list[:2], kw)  # warm-up
        sv.reset()
        t0 = time.perf_counter()
        _, rs = sv.solve_rho_s(m["rho0"], t_list, kw)
        el = time.perf_counter() - t0
        st = sv.stats()
        st_ms, st_b = _stage_stats(L, sv, reps)
        r = {"time_to_rho_s_ms": 1e3 * el, "stage_us": 1e3 * st_ms,
             "rhs_evals": evaluations(st) if isinstance(solver, H.rkdp) else st["n_rhs"],
             "bytes_per_stage": st_b}
        if cpu:
            o = O.Oracle(okind, m["N"], 0, n_threads=1).load(m)
            t0 = time.perf_counter()
            _, rs_o, _, _, _ = o.solve(m["rho0"], t_list, oracle_solver, kw["dt"],
                                       kw.get("atol", 0.0), kw.get("rtol", 0.0))
            r["cpu_oracle_ms_1_core"] = 1e3 * (time.perf_counter() - t0)
            r["rho_max_abs_diff_vs_oracle"] = float(np.abs(rs - rs_o).max())
        return r

    m = configs.exciton_chain7(max_depth=0)
    m["rho0"] = m["rho0"][:49].copy()
    kw = {"dt": m["dt"], "atol": m["atol"], "rtol": m["rtol"]}
    for form, cls, ok in (("hilb", H.redfield_hilb, O.REDFIELD_HILB),
                          ("liou", H.redfield_liou, O.REDFIELD_LIOU)):
        out["chain7_%s" % form] = timed(cls().load(m, eng), H.rkdp(), m,
                                        np.ascontiguousarray(m["t_list"]), kw, ok, O.RKDP)
    out["chain7_workload"] = ("7-site chain, 7 Drude baths (1 Drude + 2 Pade), Dormand-Prince "
                              "rtol=1e-8 atol=1e-11, t=0..1000 fs, rho every 10 fs")
    m = configs.spin_boson(max_depth=0)
    m["rho0"] = m["rho0"][:4].copy()
    out["spin_boson_hilb"] = timed(H.redfield_hilb().load(m, eng), H.rk4(), m,
                                   np.ascontiguousarray(m["t_list"]), {"dt": m["dt"]},
                                   O.REDFIELD_HILB, O.RK4)
    out["spin_boson_workload"] = "spin-boson N=2, Drude bath, RK4 dt=0.01 x 2000, rho every 10 steps"
    m = configs.dense64(max_depth=0, t_final=20.0)
    m["rho0"] = m["rho0"][:64 * 64].copy()
    kw = {"dt": m["dt"], "atol": m["atol"], "rtol": m["rtol"]}
    out["dense64_hilb"] = timed(H.redfield_hilb().load(m, eng), H.rkdp(), m,
                                np.ascontiguousarray(m["t_list"]), kw, O.REDFIELD_HILB, O.RKDP)
    out["dense64_workload"] = ("N=64 GOE H, 4 diagonal-projector baths x (1 Drude + 3 Pade), "
                               "Dormand-Prince rtol=1e-6 to t=20 (two-pass Hilbert kernels)")
    return out


def profile_stages(H, name, reps, dtype="complex128"):
    """One configuration's stage kernels only (for rocprofv3 counter passes):
    the 7-site chain (Dormand-Prince, 12650 ADOs), the N=64 dense config
    (Dormand-Prince, 969 ADOs), in `dtype` (complex128, complex64 or
    complex64_bf16x3), or the 512-member sweep (RK4, one batch, complex64
    operator then FP64), every kernel launched directly."""
    from libheom_amd import _capi, configs
    L = _capi.load()
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    eng = H.hip(0)
    if name == "sweep512":
        ms = configs.batched_sweep()
        for dtype in ("complex64", "complex128"):
            b = H.heom_batch([H.heom_hilb(m["max_depth"], dtype=dtype).load(m, eng) for m in ms])
            sv = H.qme_solver(eng, b, H.rk4())
            sv.set_graphs(False)
            _, _ = sv.solve_rho_s(b.pack([m["rho0"] for m in ms]), ms[0]["t_list"][:2],
                                  {"dt": ms[0]["dt"]})
            ns = ctypes.c_int()
            sms, sby = np.zeros(8), np.zeros(8)
            _capi.check(L.heom_solver_time_stages(sv._s, reps, p(sms), ctypes.byref(ns)))
            _capi.check(L.heom_solver_stage_bytes(sv._s, p(sby), ctypes.byref(ns)))
            n = ns.value
            print(json.dumps({"config": name, "dtype": dtype, "n_hrchy": b.n_hrchy,
                              "stage_us": [1e3 * x for x in sms[:n]],
                              "stage_bytes": [float(x) for x in sby[:n]]}))
        return
    m = configs.exciton_chain7(t_final=20.0) if name == "7site" else configs.dense64(t_final=0.2)
    q = H.heom_hilb(m["max_depth"], dtype=dtype).load(m, eng)
    sv = H.qme_solver(eng, q, H.rkdp())
    sv.set_graphs(False)
    sv.solve_rho_s(m["rho0"], m["t_list"][:2], {"dt": m["dt"], "atol": m["atol"], "rtol": m["rtol"]})
    ns = ctypes.c_int()
    ms, by = np.zeros(8), np.zeros(8)
    _capi.check(L.heom_solver_time_stages(sv._s, reps, p(ms), ctypes.byref(ns)))
    _capi.check(L.heom_solver_stage_bytes(sv._s, p(by), ctypes.byref(ns)))
    n = ns.value
    print(json.dumps({"config": name, "n_hrchy": q.n_hrchy, "stage_us": [1e3 * x for x in ms[:n]],
                      "stage_bytes": [float(x) for x in by[:n]]}))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-sweep", action="store_true")
    ap.add_argument("--no-dense", action="store_true")
    ap.add_argument("--no-spin", action="store_true")
    ap.add_argument("--no-redfield", action="store_true")
    ap.add_argument("--no-graphs", action="store_true",
                    help="launch every stage kernel directly (profiler runs)")
    ap.add_argument("--reps", type=int, default=20)
    ap.add_argument("--t-final", type=float, default=1000.0,
                    help="propagation length in fs (profiling runs use a shorter one)")
    ap.add_argument("--profile-config", choices=["7site", "dense64", "sweep512"],
                    help="counter runs: set up one configuration, run one short solve and "
                         "--reps timed passes of every stage kernel, print the stage times "
                         "and exit")
    ap.add_argument("--profile-dtype", default="complex128",
                    choices=["complex128", "complex64", "complex64_bf16x3"],
                    help="state type of --profile-config 7site / dense64")
    ap.add_argument("--summarize-trace", metavar="DB",
                    help="print a table of a rocprofv3 --kernel-trace run (*_results.db) and "
                         "exit")
    ap.add_argument("--summarize-pmc", nargs=2, metavar=("FETCH", "WRITE"),
                    help="HBM traffic of the stage kernel from two rocprofv3 --pmc runs "
                         "(their *_results.db or counter_collection.csv) of --profile-config "
                         "--pmc-config; for 7site also written to " + TRAFFIC_JSON)
    ap.add_argument("--pmc-config", choices=["7site", "dense64", "sweep512"], default="7site")
    args = ap.parse_args()
    global GRAPHS
    GRAPHS = not args.no_graphs
    if args.summarize_trace:
        print(summarize_trace(args.summarize_trace))
        return
    if args.summarize_pmc:
        from libheom_amd import configs as _c
        f, w = args.summarize_pmc
        if args.pmc_config == "7site":
            m0 = _c.exciton_chain7(t_final=10.0)
            t = summarize_pmc(f, w, m0["rho0"].nbytes)
            json.dump(t, open(TRAFFIC_JSON, "w"), indent=1)
        elif args.pmc_config == "dense64":
            m0 = _c.dense64(t_final=0.2)
            t = summarize_pmc(f, w, m0["rho0"].nbytes, kernel="hilb_mfma_kernel<64, double")
        else:
            nb = sum(m["rho0"].nbytes for m in _c.batched_sweep())
            t = {k: summarize_pmc(f, w, nb, kernel="batch_kernel<%s" % k)
                 for k in ("float", "double")}
        print(json.dumps(t))
        return
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this engine runs on one GPU; multi-GPU runs are not provided "
              "(the hierarchy is not sharded across GPUs)", file=sys.stderr)
        sys.exit(2)

    import libheom_amd as H
    from libheom_amd import _capi, configs

    if args.profile_config:
        profile_stages(H, args.profile_config, args.reps, args.profile_dtype)
        return

    m = configs.exciton_chain7(t_final=args.t_final)
    eng = H.hip(0)
    qme = H.heom_hilb(m["max_depth"]).load(m, eng)
    solver = mk_solver(H, eng, qme, H.rkdp())
    qme32 = H.heom_hilb(m["max_depth"], dtype="complex64").load(m, eng)
    solver32 = mk_solver(H, eng, qme32, H.rkdp())
    L = _capi.load()
    kw = (m["dt"], m["atol"], m["rtol"])
    t_list = np.ascontiguousarray(m["t_list"])
    nb = m["rho0"].nbytes
    d = ctypes.c_void_p()
    _capi.check(L.heom_dev_alloc(ctypes.byref(d), nb))
    rs = np.zeros((t_list.size, 7, 7), np.complex128)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)

    def one_step(sv=solver, out_rs=rs):
        sv.reset()
        _capi.check(L.heom_memcpy_h2d(d, p(m["rho0"]), nb))
        _capi.check(L.heom_device_sync())
        t0 = time.perf_counter()
        _capi.check(L.heom_solve_dev(sv._s, d, p(t_list), t_list.size, kw[0], kw[1],
                                     kw[2], p(out_rs)))
        _capi.check(L.heom_device_sync())
        return time.perf_counter() - t0, sv.stats()

    for _ in range(args.warmup):
        one_step()
    times, updates, rhs = [], 0, 0
    for _ in range(args.steps):
        el, st = one_step()
        times.append(el)
        updates += qme.n_hrchy * evaluations(st)
        rhs += evaluations(st)
    total = sum(times)
    value = updates / total

    # complex64 variant: FP32 operator and stage inputs, FP64 state, stage
    # combination and error norm; its rho_S error is taken against the FP64 run
    rs32 = np.zeros_like(rs)
    for _ in range(args.warmup):
        one_step(solver32, rs32)
    t32, u32 = 0.0, 0
    for _ in range(args.steps):
        el, st = one_step(solver32, rs32)
        t32 += el
        u32 += qme32.n_hrchy * evaluations(st)
    variant32 = {
        "dtype": "f32 operator / f64 combination", "value": u32 / t32,
        "ms_per_step": 1e3 * t32 / args.steps,
        "rho_s_max_abs_err_vs_fp64": float(np.abs(rs32 - rs).max()),
        "speedup_time_to_rho_s": total / t32,
    }
    # the oracle's committed run of exactly this job (tests/golden/chain7_dopri.npz)
    gold = golden_rho_s("chain7_dopri.npz") if args.t_final == 1000.0 else None
    if gold is not None:
        variant32["rho_s_max_abs_err_vs_oracle"] = float(np.abs(rs32 - gold).max())
    # the same with the FP64 projection of rho_0 (Hermitian, initial trace) after
    # every Dormand-Prince attempt
    qme32p = H.heom_hilb(m["max_depth"], dtype="complex64", renorm_rho0=True).load(m, eng)
    solver32p = mk_solver(H, eng, qme32p, H.rkdp())
    rs32p = np.zeros_like(rs)
    for _ in range(args.warmup):
        one_step(solver32p, rs32p)
    t32p, u32p = 0.0, 0
    for _ in range(args.steps):
        el, st = one_step(solver32p, rs32p)
        t32p += el
        u32p += qme32p.n_hrchy * evaluations(st, projected=True)
    trace_err = lambda r: float(np.abs(np.trace(r, axis1=1, axis2=2) - 1.0).max())
    variant32["trace_err"] = trace_err(rs32)
    variant32p = {
        "dtype": "f32 operator / f64 combination + f64 rho_0 projection", "value": u32p / t32p,
        "ms_per_step": 1e3 * t32p / args.steps,
        "rho_s_max_abs_err_vs_fp64": float(np.abs(rs32p - rs).max()),
        "trace_err": trace_err(rs32p),
        "speedup_time_to_rho_s": total / t32p,
    }

    # the same job through the host-buffer boundary (heom_solve): PCIe-inclusive
    host = {}
    for full in (0, 1):
        solver.reset()
        rho_h = m["rho0"].copy()
        t0 = time.perf_counter()
        solver.solve(rho_h, t_list, None, {"dt": kw[0], "atol": kw[1], "rtol": kw[2]},
                     full_copy=bool(full))
        host["time_to_rho_s_ms_full_copy_%d" % full] = 1e3 * (time.perf_counter() - t0)
    host["note"] = ("heom_solve on a host state: full_copy=0 moves rho_S per output and the "
                    "state once; full_copy=1 copies the whole state per output interval "
                    "like the reference")

    # dominant kernel: per-stage device time (HIP events) and algorithmic bytes
    ns = ctypes.c_int()
    ms = np.zeros(8)
    by = np.zeros(8)
    _capi.check(L.heom_solver_time_stages(solver._s, args.reps, p(ms), ctypes.byref(ns)))
    _capi.check(L.heom_solver_stage_bytes(solver._s, p(by), ctypes.byref(ns)))
    n = ns.value
    # the six operator passes (pass 0 is the step pass)
    avg_bytes = float(by[1:n].mean())
    avg_ms = float(ms[1:n].mean())
    achieved = avg_bytes / (avg_ms * 1e-3) / 1e9
    unit_bytes = alg_bytes_per_ado_stage(qme.n_level, qme.n_dim, "rkdp")
    ref_gbs = 7 * unit_bytes * qme.n_hrchy / (float(ms[:n].sum()) * 1e-3) / 1e9
    L.heom_dev_free(d)
    # measured HBM bytes per stage dispatch (rocprofv3 FETCH_SIZE + WRITE_SIZE,
    # calibrated on a copy of known size), recorded by --summarize-pmc
    traffic = None
    if os.path.exists(TRAFFIC_JSON):
        traffic = json.load(open(TRAFFIC_JSON)).get("traffic")

    out = {
        "metric": "ADO-stage updates/s + time-to-ρ_S(t) at err≤1e-6 vs plain FP64 on 1 GPU",
        "value": value, "unit": "ADO-stage updates/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": 1e3 * total / args.steps,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic (seeded 7-site chain, default_rng(7))",
        "config": {
            "workload": "7-site exciton chain: N=7, 7 Drude baths x (1 Drude + 2 Pade) = 21 "
                        "modes, depth 4, 12650 ADOs, heom_hilb complex128, Dormand-Prince "
                        "rtol=1e-8 atol=1e-11, t=0..%g fs, rho_S every 10 fs" % args.t_final,
            "n_hrchy": qme.n_hrchy, "main_size": qme.main_size(),
            "rhs_evals_per_step": rhs // args.steps,
            "time_to_rho_s_ms": 1e3 * total / args.steps,
        },
        "roofline": {
            "bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS, "traffic": traffic,
            "kernel": "hilb_fast_kernel<7,double> (fused Dormand-Prince stage pass)",
            "note": "the six operator passes of an attempt, the bytes they must move; stage_ms "
                    "lists the step pass (dopri_step_kernel) first",
            "bytes_per_launch": avg_bytes, "avg_launch_ms": avg_ms,
            "ados_per_launch": qme.n_hrchy,
            "stage_ms": [float(x) for x in ms[:n]],
            "reference_step": {
                "note": "the bytes of the reference's seven evaluations over the time of the "
                        "attempt's seven passes",
                "bytes_per_ado_stage": unit_bytes, "gbs": ref_gbs,
                "frac": ref_gbs / HBM_PEAK_GBS},
        },
        "rho_s_max_abs_err_vs_oracle": (float(np.abs(rs - gold).max())
                                        if gold is not None else None),
        "cpu_baseline": None,
        "variants": {"complex64": variant32, "complex64_projected": variant32p,
                     "host_buffers": host},
    }
    if not args.no_spin:
        out["variants"]["spin_boson"] = bench_spin_boson(H)
    if not args.no_dense:
        out["variants"]["dense64"] = bench_dense64(H, L, 5)
    if not args.no_sweep:
        out["variants"]["batched_sweep_512"] = bench_sweep(H, L, 1, 1, 5)
    if not args.no_redfield:
        out["variants"]["redfield"] = bench_redfield(H, L, 20, cpu=not args.no_cpu)
        out["variants"]["lsrk4_vs_rk4"] = bench_lsrk4(H, L, args.reps)
    out["stream_copy"] = stream_copy_roof(L)
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(m)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
