"""The work that a program of this framework spends its time on, as cases that can be timed.

Every case goes through the public entry points of hawaiihybrid_amd.Engine:

  sf        cf_to_sf: the spectral function of one correlation function (CF)
  cf        cf_run: the ensemble CF of one or several jobs of trajectories (He-Ar, CO2-Ar, CH4-CO2)
  array     cf_array: one ensemble reweighted to satellite temperatures
  prmu      prmu: the PR/mu spectral function of R0-injected trajectories
  zimm      cf_run with Zimmermann's trick: bound pairs, every time origin
  pipnn     PipNN.eval: N2-Ar energies and dipoles of a batch of phase points
  m0        m0: the rejection sampler's zeroth moment

Sizes are those of the reference's configurations, of bench.py and of the tests.  `exact` restates
He-Ar (a central potential, so a trajectory is planar: Gauss collocation of order 16 in R, p_R and
the polar angle), the N2-Ar networks, the transform and the sampler in plain numpy / torch FP64.
The CO2-Ar and CH4-CO2 ensembles have none: the trajectories' 64-bit integration in plain torch
takes minutes, and an orbiting pair's row depends on the last bit of any arithmetic.
"""
import itertools
import math

import numpy as np
import torch

import hawaiihybrid_amd as H
from hawaiihybrid_amd import n2ar
from hawaiihybrid_amd.data.gen_pip_n2ar import DIP_GENS, DIP_REPS, PES_GENS, PES_REPS

DT = 200.0           # a.u.: the sampling time of every configuration
ALU = 5.29177210903e-11
HTOCM = 2.1947463136320e5
HKT = 4.3597447222071e-18 / 1.380649e-23

_ENGINE = []


def engine():
    """One engine per device, as a program keeps it."""
    if not _ENGINE:
        _ENGINE.append(H.Engine(0))
    return _ENGINE[0]


# ---------------------------------------------------------------------------- the cases
def listed():
    return [
        # the spectrum of a CF of the reference's usual length, after every iteration of a run:
        # the smallest call, where launches and latency count
        dict(name="sf-4096", kind="sf", n=4096),
        # a long CF (fine frequency grid)
        dict(name="sf-1048576", kind="sf", n=1 << 20),
        # He-Ar, the first configuration: 4096 trajectories at 300 K, FP64, 2048 samples
        dict(name="cf-hear-4096", kind="cf", system="hear", precision="fp64", ntraj=4096, jobs=1, L=2048, T=300.0),
        # CO2-Ar in FP64, a small request of an odd size
        dict(name="cf-co2ar-fp64-1153", kind="cf", system="co2ar", precision="fp64", ntraj=1153, jobs=1, L=1024,
             T=200.0),
        # CO2-Ar in mixed precision, one request of the second configuration's full size
        dict(name="cf-co2ar-65536", kind="cf", system="co2ar", precision="mixed", ntraj=65536, jobs=1, L=4096,
             T=200.0),
        # the same as a batch of iterations in one call (bench.py's way)
        dict(name="cf-co2ar-6x65536", kind="cf", system="co2ar", precision="mixed", ntraj=65536, jobs=6, L=4096,
             T=200.0),
        # CH4-CO2 in mixed precision (the third configuration's 300 K and 1024 samples)
        dict(name="cf-ch4co2-12289", kind="cf", system="ch4co2", precision="mixed", ntraj=12289, jobs=1, L=1024,
             T=300.0),
        # CORRELATION_ARRAY: one He-Ar ensemble, both halves, eight satellite temperatures
        dict(name="array-hear-20000x8", kind="array", ntraj=20000, L=1024, T=300.0, ntemp=8),
        # PR/mu spectral function of He-Ar
        dict(name="prmu-hear-3000", kind="prmu", ntraj=3000, L=8192, T=300.0, R0=20.0),
        # bound He-Ar pairs with Zimmermann's trick
        dict(name="zimm-hear-1500", kind="zimm", ntraj=1500, L=1024, T=60.0),
        # N2-Ar PIP-NN energies and dipoles: the fourth configuration's batch
        dict(name="pipnn-1048576", kind="pipnn", n=1 << 20, T=300.0),
        # a zeroth-moment request of the serving mix (10^6 .. 10^8 points)
        dict(name="m0-hear-4e6", kind="m0", npoints=4000000, nstreams=65536, T=200.0),
    ]


def _log_int(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["sf", "cf", "cf", "cf", "array", "prmu", "zimm", "pipnn", "m0"])
    if kind == "sf":
        return dict(kind="sf", n=1 << rng.randint(10, 20))
    if kind == "cf":
        system = rng.choice(["hear", "co2ar", "co2ar", "ch4co2"])
        if system == "hear":
            return dict(kind="cf", system="hear", precision="fp64", ntraj=_log_int(rng, 1024, 65536), jobs=1, L=2048,
                        T=float(rng.randint(100, 500)))
        if system == "co2ar":
            if rng.random() < 0.3:
                return dict(kind="cf", system="co2ar", precision="fp64", ntraj=_log_int(rng, 512, 8192), jobs=1,
                            L=1024, T=float(rng.randint(200, 400)))
            return dict(kind="cf", system="co2ar", precision="mixed", ntraj=rng.randint(40000, 65536),
                        jobs=rng.randint(1, 4), L=4096, T=float(rng.randint(200, 400)))
        return dict(kind="cf", system="ch4co2", precision=rng.choice(["mixed", "mixed", "fp64"]),
                    ntraj=_log_int(rng, 768, 9000), jobs=1, L=rng.choice([512, 1000, 1024]), T=300.0)
    if kind == "array":
        return dict(kind="array", ntraj=_log_int(rng, 1000, 20000), L=rng.randint(256, 1024),
                    T=float(rng.randint(150, 300)), ntemp=rng.randint(1, 12))
    if kind == "prmu":
        return dict(kind="prmu", ntraj=_log_int(rng, 300, 3000), L=1 << rng.randint(12, 14),
                    T=float(rng.randint(200, 400)), R0=20.0)
    if kind == "zimm":
        return dict(kind="zimm", ntraj=_log_int(rng, 150, 1500), L=rng.randint(256, 1024),
                    T=float(rng.randint(40, 100)))
    if kind == "pipnn":
        return dict(kind="pipnn", n=_log_int(rng, 1000, 1 << 20), T=float(rng.randint(100, 500)))
    return dict(kind="m0", npoints=_log_int(rng, 1000000, 8000000), nstreams=65536, T=float(rng.randint(100, 400)))


# ---------------------------------------------------------------------------- inputs
_SYSTEMS = {"hear": (H.he_ar, H.PESMIN_HEAR, 4.0), "co2ar": (H.co2_ar, H.PESMIN_CO2AR, 4.0),
            "ch4co2": (H.ch4_co2, H.PESMIN_CH4CO2, 4.75)}


def _ics(case, seed):
    """Initial conditions [ntraj][QP] per job, from the framework's seeded host sampler."""
    kind = case["kind"]
    if kind == "cf":
        make, pesmin, rmin = _SYSTEMS[case["system"]]
        smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, case["T"], rmin, 40.0, pesmin, 40.0)
        n, jobs = case["ntraj"], case["jobs"]
        ic = H.sample_ics(make(), smp, 1000 + seed, n * jobs)[0]
        return [np.ascontiguousarray(ic[j * n:(j + 1) * n]) for j in range(jobs)]
    if kind == "prmu":
        smp = H.Sampler(H.IC_R0_INJECT, H.PAIR_FREE, case["T"], 4.0, 40.0, H.PESMIN_HEAR, case["R0"])
    elif kind == "array":
        smp = H.Sampler(H.IC_REJECTION, H.PAIR_FREE, case["T"], 4.0, 40.0, H.PESMIN_HEAR, 0.0)
    else:
        smp = H.Sampler(H.IC_REJECTION, H.PAIR_BOUND, case["T"], 4.0, 40.0, H.PESMIN_HEAR, 0.0)
    return [H.sample_ics(H.he_ar(), smp, 1000 + seed, case["ntraj"])[0]]


def _temps(case):
    """Satellite temperatures of a free-pair ensemble: up to the base temperature."""
    return [case["T"] * (0.4 + 0.6 * (i + 1) / case["ntemp"]) for i in range(case["ntemp"])]


def _cf_samples(case, seed):
    """A noisy decaying CF in the units of the reference's files."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    t = np.arange(n)
    return 1e-33 * np.exp(-t / (0.05 * n + 100.0)) * (1.0 + 0.05 * rng.standard_normal(n))


def _points(case, seed):
    return n2ar.lab_q(n2ar.phase_points(case["n"], case["T"], seed=1000 + seed))


def prepare(case, seed):
    eng = engine()
    st = dict(case=case, eng=eng, seed=seed)
    kind = case["kind"]
    if kind == "sf":
        st["cf"] = torch.from_numpy(_cf_samples(case, seed)).cuda()
    elif kind == "pipnn":
        st["q"] = torch.from_numpy(_points(case, seed)).cuda()
        st["model"] = n2ar.PipNN(eng)
    elif kind != "m0":
        st["ics"] = [eng.to_device_soa(ic) for ic in _ics(case, seed)]
    if kind == "cf":
        mixed = case["precision"] == "mixed"
        st["system"] = _SYSTEMS[case["system"]][0]()
        st["params"] = H.cf_params(case["L"], rtol=1e-10 if mixed else 1e-12,
                                   precision=H.PREC_MIXED if mixed else H.PREC_FP64)
    elif kind == "array":
        st["params"] = H.cf_params(case["L"], halves=H.HALVES_BOTH)
    elif kind == "zimm":
        st["params"] = H.cf_params(case["L"], halves=H.HALVES_BOTH, zimmermann=True)
    elif kind == "prmu":
        st["params"] = H.PrmuParams(1e-12, 1e-12, DT, case["R0"], case["L"], case["L"] // 2 + 1, H.PREC_FP64, 0, 0)
    return st


def run(st):
    case, eng = st["case"], st["eng"]
    kind = case["kind"]
    if kind == "sf":
        cf = st["cf"].clone()          # cf_to_sf apodizes its input in place
        nu, sf, _ = eng.cf_to_sf(cf, DT)
        return dict(nu=nu, sf=sf, cf=cf)
    if kind == "cf":
        return eng.cf_run(st["system"], st["params"], st["ics"])[0]
    if kind == "array":
        cf, nstar, _ = eng.cf_array(H.he_ar(), st["params"], st["ics"][0], case["T"], H.PAIR_FREE, H.PESMIN_HEAR,
                                    _temps(case))
        return dict(cf=cf, nstar=nstar)
    if kind == "zimm":
        return eng.cf_run(H.he_ar(), st["params"], st["ics"])[0]
    if kind == "prmu":
        sf, counted, _, _ = eng.prmu(H.he_ar(), st["params"], st["ics"][0])
        return dict(sf=sf, counted=counted)
    if kind == "pipnn":
        energy, mu, _ = st["model"].eval(st["q"])
        return dict(energy=energy, dipole=mu)
    smp = H.Sampler(H.IC_REJECTION, H.PAIR_FREE, case["T"], 4.0, 40.0, H.PESMIN_HEAR, 0.0)
    m, q, _ = eng.m0(H.he_ar(), smp, 1 + 100000 * st["seed"], case["npoints"], case["nstreams"])
    return dict(m=m, q=q)


# ---------------------------------------------------------------------------- work, tolerance
# Right-hand sides per trajectory (half) that the integrator's tolerance asks for, samples per
# trajectory, and operations per right-hand side (with its share of the step), per sample
# (hawaiihybrid_amd/data/flops.json; the CH4-CO2 sample is its dipole expansion: 31802 terms).
_COST = {"hear": (1100, 620, 118 + 100, 58), "co2ar": (2400, 1180, 377 + 168, 348),
         "ch4co2": (5000, 800, 900 + 270, 2 * 31802)}


def work(case):
    kind = case["kind"]
    if kind == "sf":
        n = case["n"]
        return {"bytes": 32.0 * n, "flops": 10.0 * n * (math.log2(n) + 1)}
    if kind == "pipnn":
        # 17 and 2 x 308 polynomials, the networks' products
        return {"bytes": case["n"] * 72.0, "flops": case["n"] * (1152.0 + 2 * 2 * 8984.0 + 2 * 308 * 8.0)}
    if kind == "m0":
        return {"bytes": 16.0, "flops": case["npoints"] * 1.7 * 250.0}
    system = case.get("system", "hear")
    nrhs, ns, frhs, fs = _COST[system]
    ns = min(ns, case["L"])
    if case["L"] <= 1024 and system == "co2ar":
        nrhs = 900
    halves = 2 if kind in ("array", "zimm") else 1
    n = case["ntraj"] * case.get("jobs", 1) * halves
    qp = {"hear": 6, "co2ar": 10, "ch4co2": 16}[system]
    flops = n * (nrhs * float(frhs) + ns * float(fs))
    bytes_ = 8.0 * qp * case["ntraj"] * case.get("jobs", 1) + 8.0 * case["L"] * case.get("ntemp", 1)
    if kind == "prmu":
        flops += case["ntraj"] * 2 * 5.0 * case["L"] * math.log2(case["L"])
    if kind == "zimm":
        flops += case["ntraj"] * 3 * 5.0 * 2 * case["L"] * math.log2(2 * case["L"])
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times what the path differs from `exact` by, or, where there is none, from the
    same ensemble integrated in FP64 at a tolerance ten (FP64) or a hundred (mixed) times tighter."""
    kind = case["kind"]
    if kind == "sf":
        return {"rel": 1.5e-15}       # 3.8e-16 at 2^20 points
    if kind == "pipnn":
        return {"rel": 4e-3}          # three BF16 products: energies 1e-5, the induced dipole 1e-3
    if kind == "m0":
        return {"rel": 2e-13}         # sums of squared deviations: 3.5e-14
    if kind == "cf" and case["system"] == "co2ar":
        # 2.2e-8 in FP64, 3.5e-6 in mixed precision; orbiting (chaotic) pairs add to it on some
        # ensembles, and a correct implementation is held to 1e-4 in mixed precision
        return {"rel": 1e-6 if case["precision"] == "fp64" else 1e-4}
    if kind == "cf" and case["system"] == "ch4co2":
        return {"rel": 1e-7 if case["precision"] == "fp64" else 1e-5}     # mixed: 1.9e-6
    return {"rel": 4e-11}             # He-Ar in FP64 at rtol 1e-12: 1e-11 at most


# ---------------------------------------------------------------------------- exact values
def _hear_force(R, ell2, mu):
    """-dV/dR + L^2 / (mu R^3) of the He-Ar potential (PES-IDS/HeAr.h: Tang-Toennies)."""
    A, a1, a2, b = 0.2303058634e2, 0.163051044e1, 0.4680016e-1, 0.16274792500000e1
    C = torch.tensor([0.940835513e1, 0.165523018e3, 0.379715796e4, 0.1165179999e6, 0.466258000e7, 0.236861000e9],
                     dtype=torch.float64, device=R.device).view(6, 1, 1)
    n2 = torch.arange(6, 17, 2, dtype=torch.float64, device=R.device).view(6, 1, 1)
    x, inv = b * R, 1.0 / R
    e = torch.exp(-x)
    k = torch.arange(1, 17, dtype=torch.float64, device=R.device).view(16, 1, 1)
    terms = torch.cumprod(torch.cat([torch.ones_like(x)[None], x[None] / k]), 0)
    term, csum = terms[6::2], torch.cumsum(terms, 0)[6::2]
    ip = inv[None] ** n2
    dV = A * torch.exp(-a1 * R - a2 * R * R) * (-a1 - 2.0 * a2 * R)
    dV = dV - (C * ip * (b * e * term - n2 * (1.0 - e * csum) * inv)).sum(0)
    return ell2 / mu * inv ** 3 - dV


def _hear_dipole(R):
    return torch.exp(0.47293181 - 0.40100613 * R - 0.10292726 * R * R) - 148.55391 / R ** 7


def _gauss(s):
    c, _ = np.polynomial.legendre.leggauss(s)
    c = 0.5 * (c + 1.0)
    V = np.vander(c, s, increasing=True).T                      # V[k][j] = c_j^k
    k = np.arange(1, s + 1)
    a = np.linalg.solve(V, (c[None, :] ** k[:, None]) / k[:, None]).T    # row i: int_0^{c_i}
    b = np.linalg.solve(V, 1.0 / k)
    return a, b


def _hear_path(ic, L, Rcut, sign=1.0):
    """R and the polar angle phi of the planar motion at t = 0, dt, ..., and the number of samples
    up to and including the first beyond Rcut."""
    mu, dev = H.MU_HEAR, torch.device("cuda")
    y = torch.from_numpy(np.ascontiguousarray(ic.T)).to(dev)
    R, p = y[4].clone(), sign * y[5]
    ell2 = y[3] ** 2 + (y[1] / torch.sin(y[2])) ** 2
    ell = torch.sqrt(ell2)
    phi = torch.zeros_like(R)
    a, b = (torch.from_numpy(np.ascontiguousarray(v)).to(dev) for v in _gauss(8))
    n = R.numel()
    Rs, phis = torch.full((L, n), 1e3, dtype=torch.float64, device=dev), torch.zeros((L, n), dtype=torch.float64,
                                                                                      device=dev)
    length = torch.full((n,), L, dtype=torch.int64, device=dev)
    Rs[0], phis[0] = R, phi
    live, sweeps = torch.arange(n, device=dev), 11
    for k in range(1, L):
        Fn = _hear_force(R[None], ell2, mu).expand(8, -1).contiguous()
        pn = p[None] + DT * (a @ Fn)
        for _ in range(sweeps):
            Rn = R[None] + DT / mu * (a @ pn)
            Fn = _hear_force(Rn, ell2, mu)
            pn = p[None] + DT * (a @ Fn)
        Rn = R[None] + DT / mu * (a @ pn)
        phi = phi + DT * (b @ (ell / (mu * Rn * Rn)))
        R = R + DT / mu * (b @ pn)
        p = p + DT * (b @ _hear_force(Rn, ell2, mu))
        Rs[k, live], phis[k, live] = R, phi
        if k % 16 == 0 or k == L - 1:
            # the finished trajectories leave the batch
            past = (Rs[max(1, k - 15):k + 1, live] > Rcut)
            done = past.any(0)
            first = past.to(torch.int64).argmax(0) + max(1, k - 15)
            length[live[done]] = first[done] + 1
            keep = ~done
            if not bool(keep.any()):
                break
            live, R, p, phi, ell, ell2 = (v[keep] for v in (live, R, p, phi, ell, ell2))
            sweeps = 11 if float(R.min()) < 10.0 else 4      # the far field converges faster
    return y, Rs, phis, length


def _hear_rows(ic, L, Rcut, sign=1.0):
    """mu(0).mu(t_k) per trajectory, [L][n], zero past the trajectory's end."""
    _, Rs, phis, length = _hear_path(ic, L, Rcut, sign)
    k = torch.arange(L, device=Rs.device)[:, None]
    return torch.where(k < length[None], _hear_dipole(Rs[0])[None] * _hear_dipole(Rs) * torch.cos(phis), 0.0)


def _hear_vectors(ic, L, Rcut, sign=1.0):
    """The lab dipole [3][L][n] (zero past the end) and the lengths."""
    y, Rs, phis, length = _hear_path(ic, L, Rcut, sign)
    sT, cT, sP, cP = torch.sin(y[2]), torch.cos(y[2]), torch.sin(y[0]), torch.cos(y[0])
    e1 = torch.stack([sT * cP, sT * sP, cT])
    eT, eP = torch.stack([cT * cP, cT * sP, -sT]), torch.stack([-sP, cP, torch.zeros_like(sP)])
    e2 = eT * y[3] + eP * (y[1] / sT)
    e2 = sign * e2 / torch.linalg.norm(e2, dim=0)
    d = _hear_dipole(Rs)
    k = torch.arange(L, device=Rs.device)[:, None]
    d = torch.where(k < length[None], d, 0.0)
    return e1[:, None] * (d * torch.cos(phis))[None] + e2[:, None] * (d * torch.sin(phis))[None], length


def _hear_potential(R):
    A, a1, a2, b = 0.2303058634e2, 0.163051044e1, 0.4680016e-1, 0.16274792500000e1
    C = [0.940835513e1, 0.165523018e3, 0.379715796e4, 0.1165179999e6, 0.466258000e7, 0.236861000e9]
    x = b * R
    e = torch.exp(-x)
    V = A * torch.exp(-a1 * R - a2 * R * R)
    term, csum, k = torch.ones_like(x), torch.ones_like(x), 0
    for n in range(3, 9):
        while k < 2 * n:
            k += 1
            term = term * x / k
            csum = csum + term
        V = V - C[n - 3] * (1.0 - e * csum) / R ** (2 * n)
    return V


def _hear_energy(ic):
    """Kinetic plus potential energy at the initial points."""
    y = torch.from_numpy(np.ascontiguousarray(ic.T)).cuda()
    ell2 = y[3] ** 2 + (y[1] / torch.sin(y[2])) ** 2
    return y[5] ** 2 / (2 * H.MU_HEAR) + ell2 / (2 * H.MU_HEAR * y[4] ** 2) + _hear_potential(y[4])


def _connes(n):
    r = np.arange(n) / n
    return (1.0 - r * r) ** 2


def _exact_sf(case, seed):
    n = case["n"]
    cf = _cf_samples(case, seed) * _connes(n)
    # sf_k = tmax / pi Yscale (1 / 2n) Re sum_j z_j e^{+2 pi i jk / 2n}: a DCT-III of the window's CF
    j = np.arange(2 * n)
    v = np.concatenate([cf, [0.0], -cf[:0:-1]])
    z = np.fft.ifft(v * np.exp(1j * np.pi * j / (2 * n)))[:n]
    tmax = n * DT
    atu = 2.4188843265857e-17
    yscale = atu * 8.4783536255e-30 ** 2 / (4.0 * math.pi * 8.8541878128e-12)
    nu = np.arange(n) * math.pi / tmax / 2.99792458e10 / atu / 2.0 / math.pi
    return dict(nu=nu, sf=z.real * tmax / math.pi * yscale, cf=cf)


def _exact_array(case, seed):
    ic = _ics(case, seed)[0]
    crln = 0.5 * (_hear_rows(ic, case["L"], 40.0) + _hear_rows(ic, case["L"], 40.0, -1.0)) * ALU ** 3
    E = _hear_energy(ic)
    Tb = case["T"]
    w = torch.stack([torch.exp(-E * HKT / Tb / T * (Tb - T)) for T in _temps(case)])
    for i, T in enumerate(_temps(case)):
        if T > Tb:
            w[i] = 0.0
    ns = w.sum(1)
    return dict(cf=(w @ crln.T) / ns[:, None], nstar=ns.cpu().numpy())


def _exact_prmu(case, seed):
    ic = _ics(case, seed)[0]
    L, R0 = case["L"], case["R0"]
    d, length = _hear_vectors(ic, L + 2, R0)
    counted = length <= L + 1
    # the series starts at t = dt; the sample past R0 is its last
    x = d[:, 1:L + 1] * torch.from_numpy(_connes(L)).cuda()[None, :, None]
    coeff = 4.3597447222071e-18 * ALU ** 6 * 2.4188843265857e-17 * R0 * R0 * DT * DT
    w = torch.from_numpy(-ic[:, 5] / H.MU_HEAR * coeff).cuda() * counted
    sf = torch.zeros(L // 2 + 1, dtype=torch.float64, device="cuda")
    for c in range(3):
        for t in range(0, x.shape[2], 500):
            X = torch.fft.rfft(x[c, :, t:t + 500], dim=0)
            sf += (X.real ** 2 + X.imag ** 2) @ w[t:t + 500]
    return dict(sf=sf, counted=counted.to(torch.int32).cpu().numpy())


def _exact_zimm(case, seed):
    ic = _ics(case, seed)[0]
    L = case["L"]
    df, _ = _hear_vectors(ic, L, 40.0)
    db, _ = _hear_vectors(ic, L, 40.0, -1.0)
    d = torch.cat([db.flip(1)[:, :-1], df], 1)             # series index 0 .. 2L - 2
    P = 1 << (2 * L - 1).bit_length()
    cf = torch.zeros(L, dtype=torch.float64, device="cuda")
    for c in range(3):
        a = torch.fft.rfft(d[c, :L], n=P, dim=0)
        s = torch.fft.rfft(d[c], n=P, dim=0)
        cf += torch.fft.irfft((a.conj() * s).sum(1), n=P)[:L]
    return [cf * ALU ** 3 / L / ic.shape[0]]


def _orbits(n, reps, gens):
    """The monomials (tuples of distance indices) of every polynomial: the orbit of its
    representative under the group that the generators span."""
    pair = {p: k for k, p in enumerate(itertools.combinations(range(n), 2))}
    group, todo = {tuple(range(n))}, [tuple(range(n))]
    while todo:
        g = todo.pop()
        for s in gens:
            h = tuple(s[i] for i in g)
            if h not in group:
                group.add(h)
                todo.append(h)
    perms = [[pair[tuple(sorted((g[i], g[j])))] for i, j in sorted(pair, key=pair.get)] for g in group]
    out = []
    for rep in reps.split():
        mono = () if rep == "-" else tuple(int(ch) for ch in rep)
        out.append(sorted({tuple(sorted(p[i] for i in mono)) for p in perms}) if mono else [])
    return out


def _polynomials(y, orbits):
    cache, cols = {}, []

    def mono(m):
        if m not in cache:
            cache[m] = y[m[0]] if len(m) == 1 else mono(m[:-1]) * y[m[-1]]
        return cache[m]

    for orbit in orbits:
        cols.append(sum(mono(m) for m in orbit) if orbit else torch.zeros_like(y[0]))
    return torch.stack(cols, 1)


def _mlp(x, layers):
    for k, (W, b) in enumerate(layers):
        x = x @ torch.from_numpy(W).cuda() + torch.from_numpy(b).cuda()
        if k + 1 < len(layers):
            x = x * torch.sigmoid(x)
    return x


def _quintic(x, a, b):
    r = ((x - a) / (b - a)).clamp(0.0, 1.0)
    return r * r * r * (10.0 - 15.0 * r + 6.0 * r * r)


def _exact_pipnn(case, seed):
    q = torch.from_numpy(_points(case, seed)).cuda()
    weights = n2ar.load_weights()
    half = 0.5 * H.L_N2
    pes_orbits = _orbits(3, PES_REPS, PES_GENS)
    dip_orbits = [_orbits(5, reps, gens) for reps, gens in zip(DIP_REPS, DIP_GENS)]
    E, MU = [], []
    for part in torch.split(q, 1 << 16, dim=1):
        Phi, Theta, R, p1, t1 = part
        Rh = torch.stack([torch.sin(Theta) * torch.cos(Phi), torch.sin(Theta) * torch.sin(Phi), torch.cos(Theta)])
        u = torch.stack([torch.sin(t1) * torch.cos(p1), torch.sin(t1) * torch.sin(p1), torch.cos(t1)])
        c = (Rh * u).sum(0)
        ex = u - c * Rh
        s = torch.linalg.norm(ex, dim=0)
        ex = ex / s
        ones = torch.ones_like(R)
        y = [math.exp(-0.5 * H.L_N2) * ones]
        for sign in (1.0, -1.0):
            r = torch.linalg.norm(R * Rh - sign * half * u, dim=0)
            w = _quintic(r, 6.0, 20.0)
            y.append((1.0 - w) * torch.exp(-0.5 * r) + w * 1e4 / r ** 6)
        layers, xm, xs, ym, ys = weights["pes"]
        x = (_polynomials(y, pes_orbits) - torch.from_numpy(xm).cuda()) / torch.from_numpy(xs).cuda()
        E.append((ys * _mlp(x, layers)[:, 0] + ym - n2ar.PES_EN_INF) / HTOCM)
        sites = [(half * s, half * c), (-half * s, -half * c), (half * c, -half * s), (-half * c, half * s),
                 (0.0 * ones, R)]
        w = _quintic(R, 9.5, 12.5)
        dx, dz = torch.zeros_like(R), torch.zeros_like(R)
        for (subnets, xm, xs), a0, wm in zip(weights["dip"], (2.0, 6.0), (1.0 - w, w)):
            y = [torch.exp(-torch.hypot(a[0] - b[0], a[1] - b[1]) / a0)
                 for a, b in itertools.combinations(sites, 2)]
            p = torch.cat([_polynomials(y, o) for o in dip_orbits], 1)
            xm, xs = torch.from_numpy(xm).cuda(), torch.from_numpy(xs).cuda()
            charges, at = [], 0
            for net in subnets:
                k = net[0][0].shape[0]
                ref = _mlp((-xm / xs)[None, at:at + k], net)
                charges.append(_mlp(((p - xm) / xs)[:, at:at + k], net) - ref)
                at += k
            charges = torch.cat(charges, 1)
            dx += wm * sum(charges[:, i] * sites[i][0] for i in range(5))
            dz += wm * sum(charges[:, i] * sites[i][1] for i in range(5))
        MU.append(dz * Rh + dx * ex)
    return dict(energy=torch.cat(E), dipole=torch.cat(MU, 1))


def _exact_m0(case, seed):
    """calculate_M0 on independent Mersenne Twister streams, all streams at once: a candidate takes
    ten draws (R, Phi, Theta, three normals of two, the acceptance)."""
    ns, npts, T = case["nstreams"], case["npoints"], case["T"]
    dev, M32 = torch.device("cuda"), 0xffffffff
    v = (1 + 100000 * seed + torch.arange(ns, device=dev, dtype=torch.int64)) & M32
    state = torch.empty((624, ns), dtype=torch.int64, device=dev)
    for i in range(624):
        state[i] = v
        v = (69069 * v) & M32
    quota = torch.full((ns,), npts // ns, dtype=torch.int64, device=dev)
    quota[:npts % ns] += 1
    n = torch.zeros(ns, dtype=torch.int64, device=dev)
    s1, s2 = torch.zeros(ns, dtype=torch.float64, device=dev), torch.zeros(ns, dtype=torch.float64, device=dev)
    Rmin3, Rmax3 = 4.0 ** 3, 40.0 ** 3
    kT = math.sqrt(H.MU_HEAR / HKT * T)
    bound = 1.5 * math.exp(-H.PESMIN_HEAR * HKT / T)
    rest = torch.empty((0, ns), dtype=torch.float64, device=dev)

    def twist(st):
        for i in range(624):
            yv = (st[i] & 0x80000000) | (st[(i + 1) % 624] & 0x7fffffff)
            st[i] = st[(i + 397) % 624] ^ (yv >> 1) ^ ((yv & 1) * 0x9908b0df)

    shift = None
    while bool((n < quota).any()):
        twist(state)
        w = state.clone()
        w ^= w >> 11
        w ^= (w << 7) & 0x9d2c5680
        w ^= (w << 15) & 0xefc60000
        w ^= w >> 18
        u = torch.cat([rest, w.to(torch.float64) / 4294967296.0])
        full = u.shape[0] // 10
        for k in range(full):
            d = u[10 * k:10 * k + 10]
            R = (d[0] * (Rmax3 - Rmin3) + Rmin3) ** (1.0 / 3.0)
            x = [torch.sqrt(-2 * torch.log(d[3 + 2 * i])) * torch.cos(2.0 * math.pi * d[4 + 2 * i]) for i in range(3)]
            K = kT * kT * (x[0] ** 2 + x[1] ** 2 + x[2] ** 2) / (2.0 * H.MU_HEAR)
            V = _hear_potential(R)
            weight = torch.exp(-(K + V) * HKT / T) / torch.exp(-K * HKT / T) / bound
            ok = (weight >= d[9]) & (K + V >= 0.0) & (n < quota)
            f = _hear_dipole(R) ** 2
            if shift is None:
                shift = float(f.mean()) * 0.1
            s1 += torch.where(ok, f - shift, 0.0)
            s2 += torch.where(ok, (f - shift) ** 2, 0.0)
            n += ok
        rest = u[10 * full:]
    nf = n.to(torch.float64)
    mean = s1 / nf + shift
    qs = s2 - s1 * s1 / nf
    zero_coeff = 0.00361479637 / (4.0 * math.pi)
    n0 = float(quota[0])
    return dict(m=float(mean.mean()) * zero_coeff,
                q=math.sqrt(float(qs.mean()) / n0 / (n0 - 1)) * zero_coeff)


def exact(case, seed):
    kind = case["kind"]
    if kind == "sf":
        return _exact_sf(case, seed)
    if kind == "array":
        return _exact_array(case, seed)
    if kind == "prmu":
        return _exact_prmu(case, seed)
    if kind == "zimm":
        return _exact_zimm(case, seed)
    if kind == "pipnn":
        return _exact_pipnn(case, seed)
    if kind == "m0":
        return _exact_m0(case, seed)
    if case["system"] == "hear":
        return [_hear_rows(ic, case["L"], 40.0).mean(1) * ALU ** 3 for ic in _ics(case, seed)]
    return None
