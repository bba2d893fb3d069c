"""Benchmark: IP-Glasma events/s on one MI355X, batched vs one launch
sequence per event, Pb+Pb at N=512, FP64.

A "step" is one pass of the hot path over one batch of synthetic events:
nucleons -> colour charge -> Wilson lines (Ny=50 FFT Poisson solves) ->
tau=0 root finder -> 69 leapfrog steps -> T^{mu nu} -> dE/deta, for every
event of the batch, timed from the host.  Inputs are generated on the device
(counter-based colour-charge normals); the Q_s table is resident.

Printed JSON fields beyond metric, value, unit, steps, config and the timing keys:
  plain_events_per_s  one launch sequence per event (same events, same code)
  batched_over_plain  the ratio
  roofline            the leapfrog step kernel: 1728 algorithmic bytes per
                      site-step (read+write Ux, Uy, E1, E2, phi, pi once),
                      HIP-event timed on the library's stream
  heterogeneous_batch 64 events of four collision systems and three lattice
                      sizes, batched against plain
  small_events        64 p+Pb events at N=128, batched against plain: where one
                      event leaves most of the GPU idle and the plain path is
                      bound by launch latency
  adjoint             reverse mode to rho against the forward event, Au+Au
                      N=256 and Pb+Pb N=512 (adjoint_pbpb_n512)
  large_batched_adjoint  8 Pb+Pb N=1024 Ny=100 events, one batched backward
                      per loss, events/s forward+backward and peak memory
  gluon_spectra       the evolution with the Coulomb gauge fix and spectra
                      after steps 1 and itmax, against the plain evolution
  cpu_baseline        the C oracle (OpenMP, the host's threads) on whole
                      events per phase, median of 3, at Pb+Pb N=512 (the
                      value) and Au+Au N=256, with the CPU model
"""
import argparse
import hashlib
import json
import os
import re
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "tests"))

HBM_PEAK_GBS = 8000.0
BYTES_PER_SITE_STEP = 1728
UNIQUE_BYTES_PER_SITE_STEP = 1152


def pbpb_params(I, N=512, L=30.0, Ny=50, seed=1):
    p = I.default_params()
    p.set(size=N, Ny=Ny, L=L, g=2.0, m=0.2, BG=4.0, UVdamp=0.0, QsmuRatio=0.8, rmax=1e7, roots=5020.0,
          Rapidity=0.0, useFluctuatingx=1, xFromThisFactorTimesQs=1.0, SigmaNN=70.0, maxtime=0.4,
          Projectile="Pb", Target="Pb", setWSDeformParams=1, R_WS=6.62, a_WS=0.546, beta2=0.0,
          beta3=0.0, beta4=0.0, gamma=0.0, force_dmin_flag=0, d_min=0.9, dR_np=0.0, da_np=0.0,
          bmin=0.0, bmax=0.0, samplebFromLinearDistribution=1, rotateReactionPlane=1,
          gaussianWounding=1, computeGluonMultiplicity=0, writeOutputs=0, useTimeForSeed=0,
          seed=seed, minimumQs2ST=0)
    return p


def hetero_params(I):
    """The heterogeneous batch: 16 p+Pb (N=256, L=10 fm, b in [0,5] fm),
    16 O+O (N=256, L=15 fm, Woods-Saxon R=2.61 fm, a=0.513 fm), 24 Pb+Pb
    (N=512, L=30 fm, b in [0,12] fm), 8 Pb+Pb (N=768, L=30 fm); Ny=50,
    tau_max=0.4 fm/c, FP64, one seed per event."""
    def mk(N, L, pr, tg, R, a, bmax):
        p = pbpb_params(I, N=N, L=L)
        p.set(Projectile=pr, Target=tg, R_WS=R, a_WS=a, bmin=0.0, bmax=bmax, samplebFromLinearDistribution=0)
        return p
    return ([mk(256, 10.0, "p", "Pb", 6.62, 0.546, 5.0)] * 16 + [mk(256, 15.0, "O", "O", 2.61, 0.513, 0.0)] * 16 +
            [mk(512, 30.0, "Pb", "Pb", 6.62, 0.546, 12.0)] * 24 + [mk(768, 30.0, "Pb", "Pb", 6.62, 0.546, 0.0)] * 8)


def small_params(I):
    """64 p+Pb events, N=128, L=10 fm, b in [0,5] fm, Ny=50, tau_max=0.4 fm/c."""
    p = pbpb_params(I, N=128, L=10.0)
    p.set(Projectile="p", Target="Pb", bmin=0.0, bmax=5.0, samplebFromLinearDistribution=0)
    return [p] * 64


def batch_vs_plain(I, ps, seeds, label):
    """Batched against plain over one set of events, after untimed batches
    until the autotuner has decided this batch's variants."""
    for _ in range(10):
        run_batched(I, ps, seeds)
        if all(v["chosen"] is not None for v in I.autotune_report().values()):
            break
    dtb, ob = run_batched(I, ps, seeds)
    print(f"[bench] {label} batched: {dtb:.3f} s for {len(ps)} events", file=sys.stderr, flush=True)
    dtp, op = run_plain(I, ps, seeds)
    print(f"[bench] {label} plain: {dtp:.3f} s for {len(ps)} events", file=sys.stderr, flush=True)
    rel = max(abs(x["dEdeta"] - y["dEdeta"]) / abs(y["dEdeta"]) for x, y in zip(ob, op))
    return {"events": len(ps), "batched_events_per_s": round(len(ps) / dtb, 3),
            "plain_events_per_s": round(len(ps) / dtp, 3), "batched_over_plain": round(dtp / dtb, 3),
            "batched_vs_plain_max_rel_dEdeta": rel}


def adjoint_timing(I, seed=77, system="AuAu", N=256):
    """Au+Au b=5 fm, N=256, L=30 fm, Ny=50, tau_max=0.4 fm/c (or Pb+Pb b=0 at
    N=512): one forward event (initial conditions + evolution) against the
    reverse mode to rho (initial conditions + ipg_adjoint_rho, whose forward
    pass is included)."""
    p = pbpb_params(I, N=N, L=30.0)
    if system == "AuAu":
        p.set(Projectile="Au", Target="Au", R_WS=6.38, a_WS=0.535, SigmaNN=42.0, roots=200.0, bmin=5.0, bmax=5.0)
    def timed(adj):
        ev = I.Event(p, seed=seed)
        if adj:
            # the reverse mode takes the forward's filtered colour fields
            ev.keep_slices(True)
        t0 = time.perf_counter()
        while not ev.init():
            pass
        t1 = time.perf_counter()
        if adj == "eps2":
            L, _ = ev.adjoint(loss="eps2", wrt="rho", fetch=False)
        elif adj:
            L, _ = ev.adjoint_rho(fetch=False)
        else:
            ev.run()
            L = ev.observables()["dEdeta"]
        t2 = time.perf_counter()
        if adj:
            phases[adj] = {k: round(v, 2) for k, v in ev.adjoint_phases().items() if k != "batch_init"}
        t3 = t2
        if adj:
            g = ev.rho_grad()
            t3 = time.perf_counter()
            if not np.all(np.isfinite(g)):
                raise RuntimeError("non-finite rho gradient")
        ev.close()
        return t1 - t0, t2 - t1, t3 - t2, L
    phases = {}
    timed(False)
    timed(True)
    timed("eps2")
    i_f, e_f, _, Lf = timed(False)
    i_a, e_a, f_a, La = timed(True)
    i_e, e_e, _, Le = timed("eps2")
    wl = ("Au+Au b=5 fm" if system == "AuAu" else "Pb+Pb b=0") + f", N={N}, L=30 fm, Ny=50, tau_max=0.4 fm/c"
    return {"workload": wl + ", d(dE/deta)/d rho and d eps_2/d rho", "itmax": p.itmax,
            "forward_ms": round(1e3 * (i_f + e_f), 2), "adjoint_ms": round(1e3 * (i_a + e_a), 2),
            "adjoint_over_forward": round((i_a + e_a) / (i_f + e_f), 2),
            "gradient_to_host_ms": round(1e3 * f_a, 2),
            "dEdeta_rel_diff": abs(La - Lf) / abs(Lf),
            "eps2_adjoint_ms": round(1e3 * (i_e + e_e), 2),
            "eps2_adjoint_over_forward": round((i_e + e_e) / (i_f + e_f), 2), "eps2": Le,
            "initial_conditions_ms": round(1e3 * i_f, 2),
            "phases_ms_dEdeta": phases.get(True), "phases_ms_eps2": phases.get("eps2")}


def large_batched_adjoint(I, reps=1):
    """8 Pb+Pb events at N=1024, L=40 fm, Ny=100, b uniform in [0,10] fm,
    tau_max=0.6 fm/c: the batched forward pass (initial conditions +
    evolution), then for dE/deta and for eps_2 the initial conditions of all
    events and one batched backward to rho (ipg_batch_adjoint, the gradients
    of all 8 events kept in HBM).  The checkpoint interval is the largest
    the device memory allows below sqrt(T)."""
    p = pbpb_params(I, N=1024, L=40.0, Ny=100)
    p.set(maxtime=0.6, bmin=0.0, bmax=10.0, samplebFromLinearDistribution=0)
    seeds = list(range(9000, 9008))
    I.release_cached_memory()
    out = {"workload": "8 Pb+Pb b in [0,10] fm, N=1024, L=40 fm, Ny=100, tau_max=0.6 fm/c "
                       f"(itmax={p.itmax}); gradient 2 x 100 x 8 x 1024^2 doubles per event"}
    for r in range(reps + 1):
        dt_f, ob = run_batched(I, [p] * 8, seeds)
        res = {}
        for loss in ("dEdeta", "eps2"):
            b = I.Batch([p] * 8, seeds)
            t0 = time.perf_counter()
            vals = b.adjoint(loss)
            dt = time.perf_counter() - t0
            peak, K = b.adjoint_info()
            phases = {k: round(v, 1) for k, v in b.adjoint_phases().items()}
            ok = True
            if r == reps:  # one event's gradient to the host (13.4 GB), outside the timing
                g = b.rho_grad(0, p.Ny, p.size ** 2)
                ok = bool(np.all(np.isfinite(g)))
                del g
            b.close()
            res[loss] = (dt, vals, peak, K, ok, phases)
            print(f"[bench] large batched adjoint {loss}: {dt:.2f} s for 8 events, K={K}, peak "
                  f"{peak / 2**30:.1f} GiB, phases (ms) {phases}", file=sys.stderr, flush=True)
        print(f"[bench] large batched forward: {dt_f:.2f} s for 8 events", file=sys.stderr, flush=True)
    I.release_cached_memory()
    dE = res["dEdeta"]
    e2 = res["eps2"]
    rel = max(abs(v - o["dEdeta"]) / abs(o["dEdeta"]) for v, o in zip(dE[1], ob))
    out.update({"forward_s": round(dt_f, 3), "forward_events_per_s": round(8 / dt_f, 3),
                "fwd_bwd_dEdeta_s": round(dE[0], 3), "fwd_bwd_dEdeta_events_per_s": round(8 / dE[0], 3),
                "fwd_bwd_eps2_s": round(e2[0], 3), "fwd_bwd_eps2_events_per_s": round(8 / e2[0], 3),
                "adjoint_over_forward_dEdeta": round(dE[0] / dt_f, 2),
                "adjoint_over_forward_eps2": round(e2[0] / dt_f, 2),
                "peak_device_memory_GiB": round(max(dE[2], e2[2]) / 2**30, 1),
                "checkpoint_interval": dE[3], "gradient_finite": dE[4] and e2[4],
                "phases_ms_dEdeta": dE[5], "phases_ms_eps2": e2[5],
                "adjoint_vs_forward_max_rel_dEdeta": rel,
                "eps2": [round(float(v), 6) for v in e2[1]]})
    return out


def gluon_spectra_timing(I, seed=3):
    """Evolution::run with computeGluonMultiplicity on one Pb+Pb b=0 event at
    N=512 (Ny=50, tau_max=0.4 fm/c): the gauge fix and the spectra after
    steps 1 and itmax (GaugeFix::FFTChi up to 4000 steps, three passes of
    Evolution::multiplicity), timed against the plain evolution"""
    p = pbpb_params(I, N=512)

    def timed(spectra):
        ev = I.Event(p, seed=seed)
        while not ev.init():
            pass
        t0 = time.perf_counter()
        m = ev.run_with_multiplicity() if spectra else None
        if not spectra:
            ev.run()
        dt = time.perf_counter() - t0
        d = ev.observables()["dEdeta"]
        ev.close()
        return dt, d, m

    # one untimed round first (code objects, the tuner, the gauge-fixing
    # graphs of a fresh context are captured inside the timed region alike)
    timed(True)
    timed(False)
    dt_m, d_m, m = timed(True)
    dt_r, d_r, _ = timed(False)
    it1, itm = 1, p.itmax
    return {"workload": f"Pb+Pb b=0, N=512, L=30 fm, Ny=50, tau_max=0.4 fm/c (itmax={p.itmax})",
            "evolution_with_spectra_ms": round(1e3 * dt_m, 2), "evolution_ms": round(1e3 * dt_r, 2),
            "gauge_steps": [m[it1]["gauge_iterations"], m[itm]["gauge_iterations"]],
            "gauge_residual": [m[it1]["gauge_residual"], m[itm]["gauge_residual"]],
            "dNdy": [m[it1]["dNdy"], m[itm]["dNdy"]], "dEdy_GeV": [m[it1]["dEdy"], m[itm]["dEdy"]],
            "mean_pt_GeV": [m[it1]["mean_pt"], m[itm]["mean_pt"]],
            "dEdeta_rel_diff_with_gauge_fix": abs(d_m - d_r) / abs(d_r)}


def run_plain(I, p, seeds):
    t0 = time.perf_counter()
    out = []
    ps = p if isinstance(p, list) else [p] * len(seeds)
    for p, s in zip(ps, seeds):
        ev = I.Event(p, seed=s)
        tries = 0
        while not ev.init():
            tries += 1
            if tries > 50:
                raise RuntimeError("event never succeeded")
        ev.run()
        out.append(ev.observables())
        ev.close()
    return time.perf_counter() - t0, out


def run_batched(I, p, seeds, use_graph=True):
    t0 = time.perf_counter()
    b = I.Batch(p if isinstance(p, list) else [p] * len(seeds), seeds)
    b.run(use_graph=use_graph)
    out = [b.observables(e) for e in range(len(seeds))]
    b.close()
    return time.perf_counter() - t0, out


TRAFFIC_PROFILE = os.path.join(ROOT, "profiles", "k_step_pbpb_n512_hbm_traffic.md")


def k_step_fingerprint():
    """Hash of k_step's source without comments and blanks: which kernel a
    committed counter figure belongs to."""
    src = open(os.path.join(ROOT, "ipglasma_amd", "csrc", "kernels_evolve.hip")).read()
    a = src.rindex("__global__", 0, src.index("void k_step("))
    body = re.sub(r"//[^\n]*", "", src[a:src.index("\n}\n", a)])
    return hashlib.sha256("".join(body.split()).encode()).hexdigest()[:16]


def measured_traffic(N):
    """HBM bytes per k_step launch from the committed FETCH_SIZE/WRITE_SIZE
    counter passes; None for other sizes, and where they counted another
    k_step than the present one."""
    if N != 512 or not os.path.exists(TRAFFIC_PROFILE):
        return None
    v = {}
    for line in open(TRAFFIC_PROFILE):
        k, _, x = line.partition(":")
        if k in ("traffic_bytes_per_launch", "traffic_kernel"):
            v[k] = x.strip()
    if v.get("traffic_kernel") != k_step_fingerprint():
        return None
    return int(v["traffic_bytes_per_launch"])


def roofline(I, p):
    # one untimed event first: the autotuner settles the step kernel's block order
    w = I.Event(p, seed=12344)
    while not w.init():
        pass
    w.run()
    w.close()
    ev = I.Event(p, seed=12345)
    while not ev.init():
        pass
    print("[bench] roofline event: initial conditions done", file=sys.stderr, flush=True)
    ev.enable_timing(True)
    ev.run()
    t = ev.timing()
    print("[bench] roofline event: evolution done", file=sys.stderr, flush=True)
    ev.close()
    S = p.size * p.size
    avg_ms = t["step_ms_total"] / max(1, t["nsteps"])
    achieved = BYTES_PER_SITE_STEP * S / (avg_ms * 1e-3) / 1e9
    traffic = measured_traffic(p.size)
    # the same launch against the bytes the Hermitian storage of E, phi, pi
    # actually moves (U: 2 x 144 B, E1, E2, phi, pi: 4 x 72 B, read + write)
    unique = UNIQUE_BYTES_PER_SITE_STEP * S / (avg_ms * 1e-3) / 1e9
    out = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
           "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": traffic,
           "kernel": "k_step", "avg_launch_ms": round(avg_ms, 5), "launches": t["nsteps"],
           "bytes_per_launch": BYTES_PER_SITE_STEP * S,
           "unique_bytes_per_launch": UNIQUE_BYTES_PER_SITE_STEP * S,
           "achieved_unique": round(unique, 1), "frac_unique": round(unique / HBM_PEAK_GBS, 4)}
    if traffic:
        counted = traffic / (avg_ms * 1e-3) / 1e9
        out["counter_GBps"] = round(counted, 1)
        out["frac_counter"] = round(counted / HBM_PEAK_GBS, 4)
    return out


def copy_probe(mib):
    """One plain device-to-device copy of known size (the runtime's copy
    kernel): what FETCH_SIZE and WRITE_SIZE read for it scales the counters
    of the other kernels."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")
    n = C.c_size_t(mib << 20)
    a, b = C.c_void_p(), C.c_void_p()
    if hip.hipMalloc(C.byref(a), n) or hip.hipMalloc(C.byref(b), n):
        raise RuntimeError("hipMalloc failed")
    hip.hipMemset(a, 0, n)
    hip.hipDeviceSynchronize()
    hip.hipMemcpy(b, a, n, 3)  # hipMemcpyDeviceToDevice
    hip.hipDeviceSynchronize()
    hip.hipFree(a)
    hip.hipFree(b)
    print(f"[bench] copy probe: {mib} MiB read + {mib} MiB written", file=sys.stderr, flush=True)


def cpu_model():
    """CPU model and logical CPU count of this host (lscpu)"""
    import subprocess
    model, ncpu = "unknown", os.cpu_count() or 1
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True, timeout=10).stdout
        for line in out.splitlines():
            k, _, v = line.partition(":")
            if k.strip() == "Model name":
                model = v.strip()
    except Exception:
        pass
    return model, ncpu


def oracle_event_phases(p, seed, tab, serial=()):
    """One full event of the C oracle, timed per phase: Glauber + g^2 mu^2 +
    statistics, the colour-charge normals (the reference's serial MT19937-64
    Gauss stream), setV (FFT Poisson solves and the Wilson-line products),
    the tau = 0 links + root finder + pi, the leapfrog, T^{mu nu} + dE/deta +
    Gauss law.  Phases named in `serial` run on one thread."""
    import ctypes as C
    import _cases as K
    import _oracle as O
    L = O.lib()
    L.orc_set_threads.argtypes = [C.c_int]
    nthr = L.orc_get_threads()
    N, S = p.size, p.size ** 2

    def threads(phase):
        L.orc_set_threads(1 if phase in serial else nthr)

    t = {}
    threads("glauber")
    t0 = time.perf_counter()
    st, nA, nB, info = K.oracle_event(p, seed)
    TpA, TpB, gA, gB = K.oracle_color_charge(p, nA, nB, tab)
    threads("stats")
    out = np.zeros(8)
    qc = K.qs_cfg(p)
    L.orc_stats(C.byref(qc), p.SigmaNN, info.Npart, p.minimumQs2ST, nA, len(nA), nB, len(nB), gA, gB, TpA, TpB, out)
    t["glauber_g2mu2_stats"] = time.perf_counter() - t0
    t0 = time.perf_counter()
    z = np.empty(2 * p.Ny * S * 8)
    L.orc_mt_fill(C.byref(st), 4, z.size, z)
    t["rho_normals"] = time.perf_counter() - t0
    threads("setv")
    V = np.zeros((2, S, 18))
    m_lat = p.m * (p.L / N) / 0.1973269718
    t0 = time.perf_counter()
    L.orc_setv(N, p.Ny, p.g, m_lat, 0.0, gA, gB, z.ctypes.data, None, 0, V.reshape(-1))
    t["setv"] = time.perf_counter() - t0
    del z
    threads("newton")
    ref = {k: np.zeros((S, 18)) for k in O.FIELDS}
    stats = np.zeros(5)
    t0 = time.perf_counter()
    L.orc_init_fields(N, p.g, V[0], V[1], 17, *[ref[k] for k in O.FIELDS], stats)
    t["links_newton_pi"] = time.perf_counter() - t0
    del V
    # T^{mu nu} alone on the tau = 0 state, then the whole Evolution::run
    # (which evaluates it once at itmax): evolution = run - T^{mu nu}
    threads("tmunu")
    T = np.zeros((10, S))
    t0 = time.perf_counter()
    L.orc_tmunu(N, p.g, p.L / N, p.dtau, p.itmax, *[ref[k] for k in O.FIELDS], T.reshape(-1))
    t_tmunu = time.perf_counter() - t0
    threads("evolve")
    obs = np.zeros(3)
    t0 = time.perf_counter()
    L.orc_run(N, p.g, p.L, p.dtau, p.itmax, *[ref[k] for k in O.FIELDS], T.reshape(-1), obs)
    t_run = time.perf_counter() - t0
    t["leapfrog"] = max(0.0, t_run - t_tmunu)
    t["tmunu_dedeta_gauss"] = t_tmunu
    L.orc_set_threads(nthr)
    t["total"] = sum(v for k, v in t.items())
    return t, obs[0]


def cpu_baseline(p, reps=3):
    """The C oracle (OpenMP, all host threads) on whole events: Au+Au b=5 fm
    at N=256 and Pb+Pb b=0 at N=512 (the bench's own workload), Ny=50,
    tau_max=0.4 fm/c, `reps` events each, median per phase; and one Au+Au
    event with the phases the reference runs on one thread (the rho draws,
    the FFTs of setV, T^{mu nu} and the statistics loop) on one thread."""
    import statistics
    import _cases as K
    import ipglasma_amd as I
    tab = K.load_table(I.QS_TABLE)
    model, ncpu = cpu_model()
    import _oracle as O
    threads = O.lib().orc_get_threads()
    res = {}
    for name, q in (("auau_n256", K.params("AuAu", N=256, Ny=50)), ("pbpb_n512", p)):
        runs = []
        for r in range(reps):
            ph, dedeta = oracle_event_phases(q, 100 + r, tab)
            runs.append(ph)
            print(f"[bench] cpu oracle {name} event {r}: {ph['total']:.2f} s", file=sys.stderr, flush=True)
        res[name] = {k: round(statistics.median(x[k] for x in runs), 3) for k in runs[0]}
    ser, _ = oracle_event_phases(K.params("AuAu", N=256, Ny=50), 100, tab, serial=("setv", "tmunu", "stats"))
    print(f"[bench] cpu oracle auau_n256 reference-serial phases: {ser['total']:.2f} s", file=sys.stderr, flush=True)
    res["auau_n256_reference_serial"] = {k: round(v, 3) for k, v in ser.items()}
    total = res["pbpb_n512"]["total"]
    return {"value": round(1.0 / total, 6), "unit": "events/s", "cores": threads, "kind": "port",
            "cpu_model": model, "host_cpus": ncpu,
            "sample": (f"C oracle (OpenMP, {threads} threads), whole events, median of {reps}: Pb+Pb b=0 N={p.size} "
                       f"Ny={p.Ny} {total:.2f} s/event (the value); Au+Au b=5 fm N=256 "
                       f"{res['auau_n256']['total']:.2f} s/event; seconds per phase in phases_s"),
            "phases_s": res,
            "serial_in_reference": ["rho_normals", "setv (FFTW)", "tmunu_dedeta_gauss (Tmunu)",
                                    "glauber_g2mu2_stats (statistics loop)"]}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--batch", type=int, default=8)
    ap.add_argument("--size", type=int, default=512)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-hetero", action="store_true",
                    help="skip the heterogeneous 64-event batch (N=256/512/768) and the 64 small events (N=128)")
    ap.add_argument("--no-adjoint", action="store_true", help="skip the reverse-mode timing")
    ap.add_argument("--no-spectra", action="store_true", help="skip the gauge fix + gluon spectra timing")
    ap.add_argument("--roofline-only", action="store_true",
                    help="run only the timed single event of the roofline figure (for rocprofv3)")
    ap.add_argument("--adjoint-only", action="store_true",
                    help="run only the reverse-mode timing (for rocprofv3)")
    ap.add_argument("--adjoint-pbpb-only", action="store_true",
                    help="run only the reverse-mode timing of Pb+Pb b=0 at N=512 (for rocprofv3)")
    ap.add_argument("--no-large-adjoint", action="store_true",
                    help="skip the batched reverse mode of 8 Pb+Pb events at N=1024, Ny=100")
    ap.add_argument("--large-adjoint-only", action="store_true",
                    help="run only the large batched reverse mode (for rocprofv3)")
    ap.add_argument("--spectra-only", action="store_true",
                    help="run only the gauge fix + gluon spectra timing (for rocprofv3)")
    ap.add_argument("--copy-probe", type=int, default=0, metavar="MIB",
                    help="also run one device copy of MIB MiB (the HBM counter calibration)")
    a = ap.parse_args()
    if a.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py runs on one GPU only: events are independent and there is no multi-GPU "
              "path (events would be dealt out to one process per GPU, with no collectives in the "
              "step)", file=sys.stderr)
        sys.exit(2)
    import ipglasma_amd as I
    p = pbpb_params(I, N=a.size)
    if a.copy_probe:
        copy_probe(a.copy_probe)
    if a.roofline_only:
        print(json.dumps(roofline(I, p)))
        return
    if a.adjoint_only:
        print(json.dumps(adjoint_timing(I)))
        return
    if a.adjoint_pbpb_only:
        print(json.dumps(adjoint_timing(I, seed=78, system="PbPb", N=512)))
        return
    if a.large_adjoint_only:
        print(json.dumps(large_batched_adjoint(I)))
        return
    if a.spectra_only:
        print(json.dumps(gluon_spectra_timing(I)))
        return
    seeds = list(range(1000, 1000 + a.batch))
    # untimed runs until the autotuner has decided every launch variant of
    # this workload (evolution schedule, site order of the step, inverse-row
    # block): each variant is timed three times on the real workload first
    tune_runs = 0
    while tune_runs < 12:
        run_batched(I, p, seeds)
        run_plain(I, p, seeds[:1])
        tune_runs += 1
        if all(v["chosen"] is not None for v in I.autotune_report().values()):
            break
    for w in range(a.warmup):
        run_batched(I, p, seeds)
        run_plain(I, p, seeds[:2])
    tb = 0.0
    tp = 0.0
    obs_b = obs_p = None
    for k in range(a.steps):
        dt, obs_b = run_batched(I, p, seeds)
        tb += dt
        print(f"[bench] batched step {k}: {dt:.3f} s for {a.batch} events", file=sys.stderr, flush=True)
    for k in range(a.steps):
        dt, obs_p = run_plain(I, p, seeds)
        tp += dt
        print(f"[bench] plain step {k}: {dt:.3f} s for {a.batch} events", file=sys.stderr, flush=True)
    ev_b = a.batch * a.steps / tb
    ev_p = a.batch * a.steps / tp
    # batched and plain must agree event by event
    maxrel = max(abs(x["dEdeta"] - y["dEdeta"]) / abs(y["dEdeta"]) for x, y in zip(obs_b, obs_p))
    hetero = small = None
    if not a.no_hetero:
        hp = hetero_params(I)
        hetero = {"workload": "16 p+Pb N=256 L=10, 16 O+O N=256 L=15, 24 Pb+Pb N=512 L=30 b<12, "
                              "8 Pb+Pb N=768 L=30; Ny=50, tau_max=0.4 fm/c"}
        hetero.update(batch_vs_plain(I, hp, list(range(5000, 5000 + len(hp))), "heterogeneous"))
        sp = small_params(I)
        small = {"workload": "64 p+Pb N=128 L=10 fm b<5 fm; Ny=50, tau_max=0.4 fm/c"}
        small.update(batch_vs_plain(I, sp, list(range(7000, 7000 + len(sp))), "small events"))
    adj = adj512 = large = None
    if not a.no_adjoint:
        adj = adjoint_timing(I)
        print(f"[bench] adjoint: {adj}", file=sys.stderr, flush=True)
        adj512 = adjoint_timing(I, seed=78, system="PbPb", N=512)
        print(f"[bench] adjoint N=512: {adj512}", file=sys.stderr, flush=True)
    if not a.no_adjoint and not a.no_large_adjoint:
        large = large_batched_adjoint(I)
        print(f"[bench] large batched adjoint: {large}", file=sys.stderr, flush=True)
    spectra = None
    if not a.no_spectra:
        spectra = gluon_spectra_timing(I)
        print(f"[bench] gluon spectra: {spectra}", file=sys.stderr, flush=True)
    rf = roofline(I, p)
    line = {
        "metric": "events/s: batched vs per-event launch, N=512 FP64, dE/deta rel err<=1e-9",
        "value": round(ev_b, 4), "unit": "events/s", "n_gpus": 1, "steps": a.steps, "warmup": a.warmup,
        "ms_per_step": round(1e3 * tb / a.steps, 3), "higher_is_better": True, "scaling": "weak",
        "autotune_runs": tune_runs,
        "vs_baseline": None, "dtype": "f64", "data": "synthetic (seeded Glauber nucleons, device normals)",
        "config": {"workload": f"Pb+Pb b=0, N={a.size}, L=30 fm, Ny=50, tau_max=0.4 fm/c "
                               f"(itmax={p.itmax}), batch of {a.batch} events",
                   "events_per_step": a.batch},
        "plain_events_per_s": round(ev_p, 4), "batched_over_plain": round(ev_b / ev_p, 3),
        "batched_vs_plain_max_rel_dEdeta": maxrel,
        "dEdeta_GeV": obs_b[0]["dEdeta"],
        "roofline": rf,
        "heterogeneous_batch": hetero,
        "small_events": small,
        "adjoint": adj,
        "adjoint_pbpb_n512": adj512,
        "large_batched_adjoint": large,
        "gluon_spectra": spectra,
        "autotune": I.autotune_report(),
    }
    if not a.no_cpu:
        line["cpu_baseline"] = cpu_baseline(p)
    print(json.dumps(line))


if __name__ == "__main__":
    main()
