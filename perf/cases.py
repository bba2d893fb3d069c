"""The performance cases of the framework: the calls its users make, from one
Landau frame of a small lattice to a batch of the headline Pb+Pb events.

  listed()              the named cases
  draw(rng)             one more case of the same ranges
  prepare(case, seed)   what a program holds before the call
  run(state)            one pass through the public entry points, its outputs
  work(case)            the bytes and operations one pass cannot do without
  exact(case, seed)     the outputs in 64 bits without this package, where the
                        inputs fix them (the Landau frame of given fluids)

Kinds of case:
  event     one event from its seed to T^{mu nu} on the host: a context, its
            initial conditions, the leapfrog, the observables
  batch     many events in one launch sequence, observables on the host
  reverse   one event forward and backward, the gradient on the host
  spectra   one event with the Coulomb gauge fix and the gluon spectra after
            steps 1 and itmax
  landau    the Landau frame and eccentricities of a device-resident T^{mu nu}
Everything is FP64, the only type the framework computes in.  The events of
one seed are drawn by the package's own generators (nucleons, colour-charge
normals), so nothing outside it says what they are: exact() has values for
the landau kind alone.
"""
import ctypes as C
import math

import numpy as np
import torch

import ipglasma_amd as I

# projectile, target, R_WS, a_WS, sigma_NN [mb], roots [GeV], b range [fm], b drawn linearly
SYSTEMS = {
    "pPb": ("p", "Pb", 6.62, 0.546, 70.0, 5020.0, (0.0, 5.0), 0),
    "OO": ("O", "O", 2.61, 0.513, 70.0, 5020.0, (0.0, 3.0), 1),
    "AuAu": ("Au", "Au", 6.38, 0.535, 42.0, 200.0, (5.0, 5.0), 1),
    "PbPb": ("Pb", "Pb", 6.62, 0.546, 70.0, 5020.0, (0.0, 0.0), 1),
}
# lattices the transforms take (2^a and 3 2^a) in the range the cases cover
SIZES = (64, 96, 128, 192, 256, 384, 512)
TAU = 0.4  # proper time of the fluids of the landau kind [fm/c]


def listed():
    return [
        # a serving loop that holds T^{mu nu} on the device and asks for the hydro variables, the smallest call
        {"name": "landau n=48", "kind": "landau", "N": 48, "L": 5.0},
        # the same at the largest lattice the call takes
        {"name": "landau n=1024", "kind": "landau", "N": 1024, "L": 40.0},
        # small-system scan, one event at a time: where launches and host work count
        {"name": "event p+Pb n=128", "kind": "event", "system": "pPb", "N": 128, "L": 10.0, "Ny": 50, "tau": 0.4},
        # the Au+Au input file of the tests
        {"name": "event Au+Au n=256", "kind": "event", "system": "AuAu", "N": 256, "L": 30.0, "Ny": 50, "tau": 0.4},
        # the benchmark's event, one launch sequence
        {"name": "event Pb+Pb n=512", "kind": "event", "system": "PbPb", "N": 512, "L": 30.0, "Ny": 50, "tau": 0.4},
        # the benchmark's small events: many events that each leave most of the device idle
        {"name": "batch 32 p+Pb n=128", "kind": "batch", "system": "pPb", "N": 128, "L": 10.0, "Ny": 50, "tau": 0.4,
         "events": 32},
        # mixed systems and sizes in one batch, ragged lattices among them
        {"name": "batch 12 mixed n=96-384", "kind": "batch", "system": "mixed", "N": 384, "L": 30.0, "Ny": 50,
         "tau": 0.4, "events": 12},
        # the headline benchmark: a batch of 8 central Pb+Pb events
        {"name": "batch 8 Pb+Pb n=512", "kind": "batch", "system": "PbPb", "N": 512, "L": 30.0, "Ny": 50, "tau": 0.4,
         "events": 8},
        # gradient of dE/deta with respect to the colour charges (an inference step), a ragged lattice
        {"name": "reverse rho p+Pb n=192", "kind": "reverse", "system": "pPb", "N": 192, "L": 10.0, "Ny": 10,
         "tau": 0.4, "loss": "dEdeta", "wrt": "rho"},
        # gradient of a weighted sum of the ten T^{mu nu} components with respect to the tau = 0 fields
        {"name": "reverse tmunu Pb+Pb n=256", "kind": "reverse", "system": "PbPb", "N": 256, "L": 15.0, "Ny": 50,
         "tau": 0.4, "loss": "tmunu", "wrt": "fields"},
        # the gradient of dE/deta on the headline lattice, in a box that the overlap of the nuclei fills
        {"name": "reverse dEdeta Pb+Pb n=512", "kind": "reverse", "system": "PbPb", "N": 512, "L": 15.0, "Ny": 50,
         "tau": 0.2, "loss": "dEdeta", "wrt": "fields"},
        # computeGluonMultiplicity: the gauge fix and the spectra beside the evolution
        {"name": "spectra O+O n=256", "kind": "spectra", "system": "OO", "N": 256, "L": 10.0, "Ny": 50, "tau": 0.4},
    ]


def draw(rng):
    kind = rng.choice(("landau", "event", "event", "batch", "batch", "reverse", "reverse", "spectra"))
    if kind == "landau":
        # any lattice, odd ones too
        N = int(round(math.exp(rng.uniform(math.log(32), math.log(1024)))))
        return {"kind": kind, "N": N, "L": round(N * rng.uniform(0.04, 0.12), 4)}
    top = {"event": 512, "batch": 384, "reverse": 384, "spectra": 384}[kind]
    N = rng.choice([n for n in SIZES if n <= top])
    a = rng.uniform(0.04, 0.08)  # lattice spacing [fm]: coarser ones leave the root finder's basin at some links
    # gradients and spectra are taken in boxes that the matter fills: in the far vacuum both are round-off noise
    wide = {"event": 30.0, "batch": 30.0, "reverse": 15.0, "spectra": 10.0}[kind]
    L = round(min(wide, max(5.0, N * a)), 3)
    system = "pPb" if L < 9 else rng.choice(("pPb", "OO")) if L < 10.5 else "PbPb"
    if wide > 15 and L > 12:
        system = "OO" if L < 18 else rng.choice(("AuAu", "PbPb"))
    c = {"kind": kind, "system": system, "N": N, "L": L, "Ny": rng.randint(10, 50), "tau": round(rng.uniform(0.2, 0.5), 3)}
    if kind == "batch":
        c["events"] = rng.randint(2, max(2, min(32, (384 * 384 * 8) // (N * N))))
    if kind == "reverse":
        c["loss"] = rng.choice(("dEdeta", "tmunu"))
        c["wrt"] = rng.choice(("rho", "fields"))
        if c["wrt"] == "rho":  # the gradient has a value per slice, site and colour
            c["Ny"] = rng.randint(3, 12)
    return c


def params_of(system, N, L, Ny, tau):
    pr, tg, R, a, sigma, roots, b, linear = SYSTEMS[system]
    return I.default_params(
        size=N, Ny=Ny, L=L, g=2.0, m=0.2, BG=4.0, UVdamp=0.0, QsmuRatio=0.8, rmax=1e7, roots=roots, Rapidity=0.0,
        useFluctuatingx=1, xFromThisFactorTimesQs=1.0, SigmaNN=sigma, maxtime=tau, Projectile=pr, Target=tg,
        setWSDeformParams=1, R_WS=R, a_WS=a, beta2=0.0, beta3=0.0, beta4=0.0, gamma=0.0, force_dmin_flag=0, d_min=0.9,
        dR_np=0.0, da_np=0.0, bmin=b[0], bmax=b[1], samplebFromLinearDistribution=linear, rotateReactionPlane=1,
        gaussianWounding=1, computeGluonMultiplicity=0, writeOutputs=0, useTimeForSeed=0, minimumQs2ST=0)


def events_of(case):
    """The (system, N, L) of each event of a case."""
    if case["system"] != "mixed":
        return [(case["system"], case["N"], case["L"])] * case.get("events", 1)
    n = case["events"] // 3
    return ([("pPb", 96, 7.5)] * n + [("OO", 192, 15.0)] * n +
            [("PbPb", case["N"], case["L"])] * (case["events"] - 2 * n))


def fluid(case, seed):
    """A fluctuating droplet, its fluid flowing outwards, with unlike
    pressures along the three axes: eps [S], u^tau, u^x, u^y, u^eta [4, S] and
    T^{mu nu} [10, S] (tau tau, x x, y y, eta eta, tau x, tau y, tau eta, x y,
    x eta, y eta) at tau = TAU, and the two colour-charge densities."""
    N = case["N"]
    tau = TAU
    g = torch.Generator(device="cuda").manual_seed(seed)

    def field(spread):
        # smooth random field: a few dozen Gaussian lumps over the lattice
        x = torch.arange(N, device="cuda", dtype=torch.float64) / N - 0.5
        c = torch.rand(3, 48, generator=g, device="cuda", dtype=torch.float64)
        lx = torch.exp(-((x[:, None] - (c[0] - 0.5) * spread) / 0.06) ** 2)
        ly = torch.exp(-((x[:, None] - (c[1] - 0.5) * spread) / 0.06) ** 2)
        return ((lx * (2 * c[2] - 1 if spread > 0.9 else c[2])) @ ly.T.contiguous()).reshape(-1)

    eps = 25.0 * field(0.5) + 1e-6
    vx, vy, ve = (0.25 * torch.tanh(field(1.0)) for _ in range(3))
    gam = 1.0 / torch.sqrt(1.0 - vx * vx - vy * vy - ve * ve)
    u = torch.stack([gam, gam * vx, gam * vy, gam * ve])  # orthonormal frame
    # T = eps u u + sum_i P_i e_i e_i with e_i the boosted axes
    P = (0.45, 0.35, 0.2)
    e = []
    for k in range(3):
        v = u[1 + k]
        e.append(torch.stack([v] + [v * u[1 + j] / (1.0 + gam) + (1.0 if j == k else 0.0) for j in range(3)]))

    def comp(m, n):
        return eps * (u[m] * u[n] + sum(P[k] * e[k][m] * e[k][n] for k in range(3)))

    order = ((0, 0), (1, 1), (2, 2), (3, 3), (0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3))
    T = torch.stack([comp(m, n) / tau ** ((m == 3) + (n == 3)) for m, n in order]).contiguous()
    u[3] /= tau
    g2 = torch.stack([0.05 * field(0.5).abs() for _ in range(2)])
    return eps, u, T, g2


def prepare(case, seed):
    if case["kind"] == "landau":
        p = I.default_params(size=case["N"], L=case["L"], maxtime=TAU, QsmuRatio=0.8)
        _, _, T, g2 = fluid(case, seed)
        land = torch.empty(15, case["N"] ** 2, device="cuda", dtype=torch.float64)
        return {"kind": "landau", "p": p, "it": p.itmax, "T": T, "g2": g2, "land": land}
    ps = [params_of(s, N, L, case["Ny"], case["tau"]) for s, N, L in events_of(case)]
    seeds = [1000 * (seed % 1000003) + k + 1 for k in range(len(ps))]
    weights = np.linspace(1.0, 0.1, 10) if case.get("loss") == "tmunu" else None
    return {"kind": case["kind"], "params": ps, "seeds": seeds, "loss": case.get("loss"), "weights": weights,
            "wrt": case.get("wrt")}


def new_event(state):
    return I.Event(state["params"][0], seed=state["seeds"][0])


def init(ev):
    # a draw without enough participants is drawn again, as the event loop does
    while not ev.init():
        pass


def summary(o):
    return np.array([o[k] for k in ("dEdeta", "averageQs", "averageQsAvg", "averageQsmin", "Tpp", "Qs2minST", "b",
                                    "Npart", "Ncoll")])


def run(state):
    kind = state["kind"]
    if kind == "landau":
        o = I.Observables()
        T, g2, land = state["T"], state["g2"], state["land"]
        rc = I.lib().ipg_landau_noalloc(C.byref(state["p"]), T.data_ptr(), g2[0].data_ptr(), g2[1].data_ptr(),
                                        state["it"], land.data_ptr(), C.byref(o))
        if rc:
            raise I.IPGError(I.lib().ipg_last_error().decode())
        return {"eps": land[0], "u": land[1:5], "pi": land[5:],
                "moments": np.array(list(o.eccentricity) + [o.Rbar, o.avg_eps, o.rms_r])}
    if kind == "batch":
        b = I.Batch(state["params"], state["seeds"])
        b.run()
        out = np.stack([summary(b.observables(e)) for e in range(b.n)])
        b.close()
        return out
    ev = new_event(state)
    if kind == "reverse":
        ev.keep_slices(state["wrt"] == "rho")
        init(ev)
        value, grad = ev.adjoint(loss=state["loss"], weights=state["weights"], wrt=state["wrt"])
        ev.close()
        return {"value": value, "grad": grad}
    init(ev)
    if kind == "spectra":
        m = ev.run_with_multiplicity()
        spectra = {str(it): {k: m[it][k] for k in ("dNdy", "dEdy", "n_kt", "E_kt", "counts")} for it in m}
        out = {"spectra": spectra, "T": ev.tmunu()}
        ev.close()
        return out
    ev.run()
    out = {"observables": summary(ev.observables()), "T": ev.tmunu()}
    ev.close()
    return out


def steps(N, L, tau):
    return int(10 * tau / (L / N)) + 1


def work(case):
    """Compulsory work.  The lattice state does not fit on chip, so a leapfrog
    step reads and writes U_x, U_y (18 doubles a site) and E1, E2, phi, pi (9)
    once: 1152 B and ~4.6 kflop a site.  A colour-charge slice of a nucleus
    goes through memory twice for its two-dimensional transforms (four
    complex fields a site written and read, twice: 256 B) and takes ~2.2 kflop
    a site (normals, transforms, the exponential).  The tau = 0 root finder
    takes ~2 iterations of ~10 kflop a link.  Backward, a step reads the
    states before and after it and reads and writes the cotangents of the six
    fields: 2.3 kB and ~14 kflop a site."""
    if case["kind"] == "landau":
        S = case["N"] ** 2
        return {"bytes": 8 * S * (10 + 2 + 15), "flops": 3000 * S}
    nbytes = flops = 0.0
    for _, N, L in events_of(case):
        S, T = N * N, steps(N, L, case["tau"])
        nbytes += S * (1152 * T + 256 * 2 * case["Ny"])
        flops += S * (4600 * T + 2200 * 2 * case["Ny"] + 2 * 2 * 10000)
        if case["kind"] == "reverse":
            nbytes += S * 2304 * T
            flops += S * 14000 * T
            if case["wrt"] == "rho":
                nbytes += S * (256 + 64) * 2 * case["Ny"]
                flops += S * 3000 * 2 * case["Ny"]
            else:
                nbytes += S * 6 * 18 * 8
        elif case["kind"] != "batch":
            nbytes += S * 80
    return {"bytes": nbytes, "flops": flops}


def exact(case, seed):
    """The fluid's own eps and u^mu (the rest frame below 0.1 fm^-4, where the
    framework sets it); pi^{mu nu} and the moments follow the reference's
    conventions and have no value here."""
    if case["kind"] != "landau":
        return None
    eps, u, _, _ = fluid(case, seed)
    rest = torch.zeros_like(u)
    rest[0] = 1.0
    return {"eps": eps, "u": torch.where(eps > 0.1, u, rest), "pi": None, "moments": None}
