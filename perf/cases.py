"""Performance cases: what a user of this framework has it do, through its
public entry points, from the smallest calls to the largest.

Six kinds of call, with the sizes and distributions of the benchmark
configurations, the served stream and the tests:

  batch     device-resident tracers advanced over a run of snapshots, the
            spectra downloaded at its end (Batch.run, batch_get_state)
  snapshot  the drop-in for the reference's per-snapshot call: host arrays in
            and out (execute_snapshot)
  serve     a burst of tracer chunks through the request loop
            (Server.submit / wait)
  solve     the batched Chang-Cooper solve on caller-owned device arrays
            (solve_cc_batch_noalloc)
  ic, had   inverse-Compton / hadronic emissivities of host spectra: the
            kernel table at this snapshot's redshift (IC) or the run's table
            (hadronic), then the contraction
  synch     synchrotron emissivities of host spectra on a pitch-kernel table,
            through the plan (MFMA mode) or the one-shot call
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "croma-fp_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import croma_hip as ch  # noqa: E402
import synth  # noqa: E402

GRIDS = (64, 128, 256, 512)
MODES = {"fp64": ch.EMIS_FP64, "fp32": ch.EMIS_FP32, "mfma": ch.EMIS_MFMA_XF32}
# mean substeps per tracer and Gyr of the synthetic backgrounds (the 1e6
# tracer configuration: 2,092 per tracer and snapshot of 0.385 Gyr)
NSUB_PER_GYR = 5400.0
FREQ = (7.0, 11.0)      # log10 Hz, synchrotron
IC_FREQ = (8.0, 28.0)   # log10 Hz, inverse Compton
LOGB = (-3.0, 6.0)      # first plane (log10 microgauss) and decades of the synchrotron table


def listed():
    return [
        # the smallest chunk of the served stream, alone: latency and launches
        dict(name="batch 256 e n64", kind="batch", n=64, ntr=256, species=1, dpp=3, nsnap=10, z0=0.1, dsa=0.0,
             window=0, cap=0.0, fp32=False, tune=False),
        # the CPU-runnable configuration: 1,024 tracers x 128 bins, D_pp off
        dict(name="batch 1024 e n128", kind="batch", n=128, ntr=1024, species=1, dpp=3, nsnap=10, z0=0.1, dsa=0.0,
             window=0, cap=0.0, fp32=False, tune=False),
        # batched uneven work: 10,000 tracers of both species, ASA, shock sources on 5%
        dict(name="batch 10000 ep n256 asa", kind="batch", n=256, ntr=10000, species=3, dpp=1, nsnap=10, z0=0.1,
             dsa=0.05, window=0, cap=0.0, fp32=False, tune=True),
        # bulk throughput: electrons on 512 bins, TTD, the largest served chunk
        dict(name="batch 65536 e n512 ttd", kind="batch", n=512, ntr=65536, species=1, dpp=2, nsnap=10, z0=0.5,
             dsa=0.0, window=0, cap=0.0, fp32=False, tune=True),
        # options in earnest: eta cap and on-window (in-kernel secondaries), an odd count
        dict(name="batch 3001 ep n128 cap", kind="batch", n=128, ntr=3001, species=3, dpp=2, nsnap=4, z0=0.04,
             dsa=0.0, window=1, cap=0.1, fp32=False, tune=False),
        # the reference's own call, once per snapshot, host arrays
        dict(name="snapshot 2000 ep n128", kind="snapshot", n=128, ntr=2000, species=3, dpp=1, z0=0.02),
        # a burst of mixed chunks through the request loop
        dict(name="serve 6 chunks", kind="serve", chunks=6, lo=256, hi=6000, nsnap=10, z0=0.2),
        # the solver alone: a handful of systems, and as many as the call takes
        dict(name="solve 64x64", kind="solve", nsys=64, nrow=64),
        dict(name="solve 8192x512", kind="solve", nsys=8192, nrow=512),
        # a snapshot's inverse-Compton emissivities: its table, then the contraction
        dict(name="ic 40000 n256 mfma", kind="ic", n=256, ntr=40000, nbins=64, mode="mfma"),
        # a snapshot's synchrotron emissivities through the plan
        dict(name="synch 20000 n256 mfma", kind="synch", n=256, ntr=20000, nbins=64, mode="mfma", planes=512),
        # and in full precision, on an odd count
        dict(name="synch 5001 n128 fp64", kind="synch", n=128, ntr=5001, nbins=48, mode="fp64", planes=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("batch", "batch", "batch", "batch", "snapshot", "serve", "solve", "solve", "ic", "had",
                       "synch"))
    n = rng.choice(GRIDS)
    if kind == "batch":
        species = rng.choice((1, 1, 3))
        # at most the largest listed case's work (species x tracers x bins x Gyr)
        nsnap = rng.randint(2, 10)
        z0 = round(rng.uniform(0.01, 0.05), 4) * nsnap
        most = min(65536, int(65536 * 512 * 0.5 * 0.9 / (n * z0 * (3.0 if species == 3 else 1.0))))
        ntr = _log_int(rng, 256, min(most, 65536 if species == 1 else 12000))
        special = species == 3 and n <= 256 and ntr < 4000 and rng.random() < 0.4
        return dict(kind=kind, n=n, ntr=ntr, species=species, dpp=rng.choice((1, 2, 3)), nsnap=nsnap, z0=z0,
                    dsa=0.05 if (species == 3 and not special and rng.random() < 0.5) else 0.0,
                    window=1 if special else 0, cap=0.1 if special else 0.0,
                    fp32=(species == 1 and rng.random() < 0.25), tune=ntr >= 8192)
    if kind == "snapshot":
        return dict(kind=kind, n=n, ntr=_log_int(rng, 100, 6000), species=rng.choice((1, 3)), dpp=rng.choice((1, 2, 3)),
                    z0=round(rng.uniform(0.01, 0.04), 4))
    if kind == "serve":
        return dict(kind=kind, chunks=rng.randint(2, 8), lo=256, hi=_log_int(rng, 1000, 6000), nsnap=10,
                    z0=round(rng.uniform(0.1, 0.3), 3))
    if kind == "solve":
        nrow = rng.choice((64, 128, 256, 512, rng.randint(3, 700)))
        return dict(kind=kind, nsys=_log_int(rng, 16, 4194304 // nrow), nrow=nrow)
    if kind in ("ic", "had"):
        n = rng.choice((64, 128, 256))
        return dict(kind=kind, n=n, ntr=_log_int(rng, 500, 40000), nbins=rng.choice((40, 64, rng.randint(10, 128))),
                    mode=rng.choice(("mfma", "mfma", "fp32", "fp64")))
    mode = rng.choice(("mfma", "mfma", "fp32", "fp64"))
    n = rng.choice((64, 128, 256))
    return dict(kind=kind, n=n, ntr=_log_int(rng, 500, 20000 if mode == "mfma" else 6000),
                nbins=rng.choice((32, 48, 64)), mode=mode, planes=512)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _axis(n, lo, hi):
    """Bin centres and widths of the momentum grid (half the distance of the neighbours)."""
    step = (hi - lo) / n
    a, p = lo - step, np.empty(n + 2)
    for j in range(n + 2):
        p[j] = 10.0 ** a
        a = a + step
    return p[1:-1], 0.5 * (p[2:] - p[:-2])


def _spectra(rng, p, ntr):
    """Power laws q ~ U(2, 3.5) with log-uniform exponential cutoffs and amplitudes."""
    q = rng.uniform(2.0, 3.5, ntr)
    cut = 10.0 ** rng.uniform(2.0, 6.0, ntr)
    amp = rng.uniform(-3.0, 3.0, ntr) * math.log(10.0)
    return np.exp(amp[:, None] - q[:, None] * np.log(p)[None, :] - p[None, :] / cut[:, None])


def _synch_table(n, nbins, planes):
    """Pitch-averaged synchrotron kernel table [plane][frequency][bin]: F(x)
    in its closed approximation 2.15 x^(1/3) (1 + x)^(1/6) e^-x, zero below
    the double range as the averaged kernel is."""
    p = _axis(n, 0.0, 6.0)[0]
    b = 10.0 ** (LOGB[0] + LOGB[1] / planes * np.arange(planes)) * 1.0e-6
    nu = 10.0 ** np.linspace(FREQ[0], FREQ[1], nbins)
    x = nu[None, :, None] / (4.194284e6 * b[:, None, None] * (1.0 + p * p)[None, None, :])
    with np.errstate(under="ignore"):
        return 2.15 * np.cbrt(x) * (1.0 + x) ** (1.0 / 6.0) * np.exp(-x)


def _workload(case, seed):
    return synth.make_workload(n=case["n"], ntracer=case["ntr"], nsnap=case.get("nsnap", 1), species=case["species"],
                               dpp_model=case["dpp"], seed=seed, z0=case["z0"], dsa_frac=case.get("dsa", 0.0))


def _params(case):
    p = dict(dpp_model=case["dpp"], tracer_nsub_safety=0.5)
    if case.get("window"):
        p["reacc_window_mode"] = 1
    if case.get("cap"):
        p["eta_dpp_cap"] = case["cap"]
    return ch.default_params(**p)


def _serve_chunks(case, seed):
    rng = np.random.default_rng(seed)
    out = []
    for i in range(case["chunks"]):
        # the mix is the case's, the backgrounds are the seed's
        mix = np.random.default_rng(1000 + i)
        ntr = int(round(10.0 ** mix.uniform(math.log10(case["lo"]), math.log10(case["hi"]))))
        n, species, dpp = int(mix.choice(GRIDS)), int(mix.choice((1, 2, 3))), int(mix.choice((1, 2, 3)))
        k = case["nsnap"]
        w = synth.make_workload(n=n, ntracer=ntr, nsnap=k + 1, species=species, dpp_model=dpp,
                                seed=int(rng.integers(1 << 30)), z0=case["z0"])
        out.append(dict(n=n, species=species, dpp_model=dpp, z=w.z[:k + 1], dt_snap=w.dt_snap[:k],
                        bg=np.ascontiguousarray(w.bg[:k + 1]), cre=w.cre0, crp=w.crp0 if w.protons else None,
                        mass=w.mass))
    return out


def _solve_systems(case, seed, device):
    """Chang-Cooper systems b x_j - a x_{j-1} - c x_{j+1}: non-negative
    couplings, b = 1 + dt / T + a + c, sources and states over many decades."""
    g = torch.Generator(device="cpu").manual_seed(seed)
    ns, nr = case["nsys"], case["nrow"]

    def u(lo, hi, shape=(ns, nr)):
        return torch.rand(shape, generator=g, dtype=torch.float64) * (hi - lo) + lo

    a = u(0.0, 2.0) * 10.0 ** u(-3.0, 2.0, (ns, 1))
    c = u(0.0, 2.0) * 10.0 ** u(-3.0, 2.0, (ns, 1))
    a[:, 0] = 0.0
    c[:, -1] = 0.0
    b = 1.0 + u(0.0, 0.1) + a + c
    q = 10.0 ** u(-6.0, 0.0)
    x = 10.0 ** u(-20.0, 0.0)
    return [t.to(device) for t in (a, b, c, q, x)]


SOLVE_DT = 0.0137


def _emission_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n, ntr, nbins = case["n"], case["ntr"], case["nbins"]
    if case["kind"] == "had":
        p = _axis(n, -1.0, 8.0)[0]
        centres = np.linspace(0.0, 7.0, nbins)
        fk = np.exp(-0.5 * ((np.log10(p)[None, :] - centres[:, None]) / 0.9) ** 2)
        return dict(spec=_spectra(rng, p, ntr), n_gas=10.0 ** rng.uniform(-5.0, -2.0, ntr), fk=fk)
    p = _axis(n, 0.0, 6.0)[0]
    if case["kind"] == "ic":
        return dict(spec=_spectra(rng, p, ntr), z=float(rng.uniform(0.0, 1.0)))
    return dict(spec=_spectra(rng, p, ntr), b=10.0 ** rng.uniform(-8.0, -5.0, ntr))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        w = _workload(case, seed)
        ctx = ch.Context(case["n"], _params(case))
        if case["fp32"]:
            ctx.set_coeff_precision(True)
        b = ch.Batch(ctx, w.ntracer, w.species, w.nsnap)
        b.set_state(w.crp0 if w.protons else None, w.cre0, mass=w.mass)
        for s in range(w.nsnap):
            b.set_background(s, w.bg[s])
            if s in w.qpi or s in w.qepri:
                b.set_sources(s, w.qpi.get(s), w.qepri.get(s))
        if case["tune"]:
            b.autotune(0, w.nsnap, w.z, w.dt_snap)
        size = case["ntr"] * case["n"]
        return dict(kind=kind, ctx=ctx, b=b, nsnap=w.nsnap, z=w.z, dt=w.dt_snap, cre=np.zeros(size),
                    crp=np.zeros(size) if w.protons else None, shape=(case["ntr"], case["n"]))
    if kind == "snapshot":
        w = _workload(case, seed)
        ctx = ch.Context(case["n"], _params(case))
        row, m1, p1 = ctx.ic_cooling_row(float(w.z[0]))
        rown, m1n, p1n = ctx.ic_cooling_row(float(w.z[1]))
        f = w.bg[0]
        ns, non = ctx.nsub(float(w.dt_snap[0]), f[0], f[1], f[2], f[3], row[0], row[-1], f[4], f[5])
        fqe, npmin = ctx.secondary_weights()
        zero = np.zeros(case["ntr"] * case["n"])
        return dict(kind=kind, ctx=ctx, ns=ns, non=non, dt=float(w.dt_snap[0]), bg0=w.bg[0], bg1=w.bg[1],
                    row=(row, m1, p1), rown=(rown, m1n, p1n), zero=zero, fqe=fqe, npmin=npmin, mass=w.mass,
                    crp=w.crp0.copy(), cre=w.cre0.copy(), shape=(case["ntr"], case["n"]))
    if kind == "serve":
        return dict(kind=kind, srv=ch.Server(16 << 30, ch.default_params(tracer_nsub_safety=0.5)),
                    chunks=_serve_chunks(case, seed))
    if kind == "solve":
        t = _solve_systems(case, seed, "cuda")
        return dict(kind=kind, t=t, out=torch.zeros_like(t[0]))
    e = _emission_inputs(case, seed)
    ctx = ch.Context(case["n"], ch.default_params())
    st = dict(kind=kind, ctx=ctx, mode=MODES[case["mode"]], nbins=case["nbins"], **e)
    if kind == "synch":
        st["table"] = _synch_table(case["n"], case["nbins"], case["planes"])
        st["tab_args"] = (case["nbins"], case["planes"], LOGB[0], case["planes"] / LOGB[1])
        st["plan"] = ch.SynchPlan(ctx, st["table"], *st["tab_args"]) if case["mode"] == "mfma" else None
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    kind = st["kind"]
    if kind == "batch":
        st["b"].run(0, st["nsnap"], st["nsnap"], st["z"], st["dt"])
        ptr = ctypes.POINTER(ctypes.c_double)
        cre, crp = st["cre"], st["crp"]
        rc = ch.lib().croma_hip_batch_get_state(ctypes.c_void_p(st["b"].h),
                                                crp.ctypes.data_as(ptr) if crp is not None else None,
                                                cre.ctypes.data_as(ptr))
        if rc:
            raise ch.CromaHipError(rc, "batch_get_state")
        out = {"cre": cre.reshape(st["shape"])}
        if crp is not None:
            out["crp"] = crp.reshape(st["shape"])
        return out
    if kind == "snapshot":
        st["ctx"].execute_snapshot(st["ns"], st["non"], True, 0.0, st["dt"], st["bg0"], *st["row"], st["bg1"],
                                   *st["rown"], st["zero"], st["zero"], st["fqe"], st["npmin"], st["mass"], None,
                                   st["crp"], st["cre"])
        return {"cre": st["cre"].reshape(st["shape"]), "crp": st["crp"].reshape(st["shape"])}
    if kind == "serve":
        ids = [st["srv"].submit(**c) for c in st["chunks"]]
        return [st["srv"].wait(i)[:2] for i in ids]
    if kind == "solve":
        t, out = st["t"], st["out"]
        ns, nr = out.shape
        ch.solve_cc_batch_noalloc(ns, nr, SOLVE_DT, *[x.data_ptr() for x in t], out.data_ptr())
        return out
    ctx = st["ctx"]
    if kind == "ic":
        fic, _ = ctx.emission_kernel_table(ch.TABLE_IC, st["nbins"], *IC_FREQ, z=st["z"])
        return {"table": fic, "eps": ctx.emission_ic(st["spec"], fic, st["nbins"], st["mode"])[0]}
    if kind == "had":
        return ctx.emission_hadronic(st["spec"], st["n_gas"], st["fk"], st["nbins"], -1.0, 5.0, st["mode"])[0]
    if st["plan"] is not None:
        return st["plan"].run(st["spec"], st["b"])[0]
    return ctx.emission_synch(st["spec"], st["b"], st["table"], *st["tab_args"], mode=st["mode"])[0]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _gyr(z0):
    return float(np.diff(synth.lcdm_age_gyr(np.array([z0, 0.0])))[0])


def work(case):
    kind = case["kind"]
    if kind in ("batch", "snapshot"):
        sp, n, ntr = (2 if case["species"] == 3 else 1), case["n"], case["ntr"]
        k = case.get("nsnap", 1)
        # spectra read and written once, the backgrounds of each snapshot read; 10 flops
        # a row and substep of each species (right-hand side, elimination, back substitution)
        return {"bytes": 16.0 * sp * ntr * n + 64.0 * ntr * k + (16.0 * ntr * n * case["dsa"] * k if case.get("dsa") else 0.0),
                "flops": 10.0 * n * sp * ntr * max(10.0 * k, NSUB_PER_GYR * _gyr(case["z0"]))}
    if kind == "serve":
        by = fl = 0.0
        for i in range(case["chunks"]):
            mix = np.random.default_rng(1000 + i)
            ntr = 10.0 ** mix.uniform(math.log10(case["lo"]), math.log10(case["hi"]))
            n, species = int(mix.choice(GRIDS)), int(mix.choice((1, 2, 3)))
            sp = 1 if species == 1 else 2
            by += 16.0 * sp * ntr * n + 64.0 * ntr * (case["nsnap"] + 1)
            fl += 10.0 * n * sp * ntr * NSUB_PER_GYR * _gyr(case["z0"])
        return {"bytes": by, "flops": fl}
    if kind == "solve":
        return {"bytes": 48.0 * case["nsys"] * case["nrow"], "flops": 10.0 * case["nsys"] * case["nrow"]}
    n, ntr, nb = case["n"], case["ntr"], case["nbins"]
    by, fl = 8.0 * ntr * (n + nb + 1), 2.0 * ntr * n * nb
    if kind == "ic":
        fl += 400.0 * 20.0 * n * nb  # 400-node quadrature per table entry
        by += 8.0 * n * nb
    if kind == "synch":
        fl += 3.0 * ntr * n * nb  # the log-linear interpolation of each kernel value
        by += 8.0 * case["planes"] * nb * n
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """About four times what another order of the sums (another launch shape)
    or the 64-bit results of exact() showed."""
    kind = case["kind"]
    if kind == "batch" and case["fp32"]:
        return {"rel": 1e-7, "max": 2.2e-6}  # FP32 coefficients: 2.5e-8 and 5.4e-7 off FP64
    if kind in ("batch", "snapshot", "serve"):
        return {"rel": 5e-14, "max": 2e-12}  # 1.2e-14 off exact(), 7e-16 and 2.2e-14 between launch shapes
    if kind == "solve":
        return {"rel": 1e-15, "max": 4e-14}
    if case["mode"] != "fp64":
        # FP32 accumulation: split-BF16 x3 up to 1.5e-6, FP32 2.6e-7
        return {"rel": 6e-6 if case["mode"] == "mfma" else 1e-6, "max": 4e-5}
    # the IC table's Wien tail cancels: 1.7e-10 and 2.6e-8 between its restatements
    return {"rel": 7e-10, "max": 1.1e-7} if kind == "ic" else {"rel": 4e-15, "max": 1e-13}


# ---------------------------------------------------------------------------
# the same results in plain 64-bit arithmetic
# ---------------------------------------------------------------------------
C_LIGHT, GEV, GYR, MP, ME = 2.999e10, 1.6e-3, 3.1536e16, 0.938, 0.511e-3
H_PL, MEG, T0, KB = 6.63e-27, 9.11e-28, 2.757, 1.38e-16


def _cmb(eps, z):
    """CMB photon density per unit energy (electron rest energies)."""
    x = eps * MEG * C_LIGHT * C_LIGHT / (KB * T0 * (1.0 + z))
    pre = 8.0 * math.pi * C_LIGHT ** 3 * (MEG / H_PL) ** 3
    with np.errstate(over="ignore", divide="ignore", invalid="ignore"):
        v = pre * eps * eps / (np.exp(np.minimum(x, 700.0)) - 1.0)
    return np.where(x > 90.0 * math.log(10.0), 0.0, v)


def _ic_sigma(e0, gamma, eps):
    with np.errstate(divide="ignore", invalid="ignore", over="ignore"):
        k = eps / (4.0 * e0 * gamma * (gamma - eps))
        kk = np.where(k > 0.0, k, 1.0)
        v = 2.0 * kk * np.log(kk) + (1.0 + 2.0 * kk) * (1.0 - kk) + (4.0 * e0 * kk * gamma) ** 2 / (
            2.0 * (1.0 + 4.0 * e0 * gamma * kk)) * (1.0 - kk)
    return np.where(k > 0.0, 2.0 * math.pi * 2.82e-13 ** 2 * C_LIGHT / (gamma * gamma * e0) * v, 0.0)


def _ic_table(n, nbins, z):
    """Inverse-Compton emissivity per electron, 400-node trapezoid over log photon energy."""
    p = _axis(n, 0.0, 6.0)[0]
    gamma = np.sqrt(1.0 + p * p)
    d = (IC_FREQ[1] - IC_FREQ[0]) / nbins
    out = np.empty((nbins, n))
    for k in range(nbins):
        eps = H_PL * 10.0 ** (IC_FREQ[0] + k * d) / (MEG * 3.0e10 ** 2)
        with np.errstate(divide="ignore"):
            lo = eps / (4.0 * gamma * (gamma - eps))
        lo = np.where(lo < 0.0, eps / (gamma * gamma), lo)
        a0, a1 = np.log10(lo), math.log10(eps)
        e0 = 10.0 ** (a0[None, :] + (a1 - a0)[None, :] / 400.0 * np.arange(401)[:, None])
        f = _ic_sigma(e0, gamma[None, :], eps) * _cmb(e0, z)
        out[k] = H_PL * eps * (0.5 * (f[1:] + f[:-1]) * np.diff(e0, axis=0)).sum(0) / (4.0 * math.pi)
    return out


def _cmb_bounds(z):
    """Photon energies where the CMB density falls to 10^-5.5 of its value at kT (Newton)."""
    delta, c, t0, m = 10.0 ** -5.5, 3.0e10, 2.725, 9.11e-28
    kt = KB / (m * c * c) * t0 * (1.0 + z)
    pre = 8.0 * math.pi * C_LIGHT ** 3 * (MEG / H_PL) ** 3
    s = MEG * C_LIGHT * C_LIGHT / (KB * T0 * (1.0 + z))
    aim = float(_cmb(np.float64(kt), z)) * delta
    got = []
    for start in (0.01, 10.0):
        eps, new = 1.0, start * kt
        while abs(new - eps) > delta * eps:
            eps = new
            em = math.exp(eps * s)
            dn = pre * eps / (em - 1.0) * (2.0 - eps * s * em / (em - 1.0))
            new = eps - (float(_cmb(np.float64(eps), z)) - aim) / dn
        got.append(new)
    return got


def _ic_row(p, z):
    """Inverse-Compton loss rate: trapezoid over the photon energy of the
    trapezoid over the scattered energy, log steps of 0.05."""
    lo, hi = _cmb_bounds(z)
    da, gamma = 0.05, np.sqrt(1.0 + p * p)
    n_out = int(round((math.log10(hi) - math.log10(lo)) / da))
    e0 = 10.0 ** (math.log10(lo) + da * np.arange(n_out + 1))
    inner = np.empty((n_out + 1, len(p)))
    for i, e in enumerate(e0):
        top = 4.0 * gamma * gamma * e / (1.0 + 4.0 * e * gamma)
        cnt = np.round((np.log10(top) - math.log10(e)) / da).astype(int)
        eps = 10.0 ** (math.log10(e) + da * np.arange(max(1, cnt.max()) + 1))
        f = eps[:, None] * _ic_sigma(e, gamma[None, :], eps[:, None])
        seg = 0.5 * (f[1:] + f[:-1]) * np.diff(eps)[:, None]
        inner[i] = np.where(np.arange(len(seg))[:, None] < cnt[None, :], seg, 0.0).sum(0)
    f = inner * _cmb(e0, z)[:, None]
    return GYR * (0.5 * (f[1:] + f[:-1]) * np.diff(e0)[:, None]).sum(0)


def _erf(x):
    return torch.erf(torch.from_numpy(np.ascontiguousarray(x))).numpy()


def _coulomb_p(n_gas, p, kbt):
    def kern(x):
        return 0.5 * math.sqrt(math.pi) * _erf(np.sqrt(x)) - np.sqrt(x) * np.exp(-x)

    g = math.sqrt(1.0 + p * p)
    xp = (g * MP - MP) / kbt
    thermal = 1.0 - kbt / (2.0 * MP * (g - 1.0))
    v = GYR * C_LIGHT / (MP * GEV) * (kern(xp * (ME / MP)) + kern(xp) * (ME / MP)) * n_gas * (1.0 + p * p) / (
        p * p) * thermal * 3.5e-29
    return np.where(thermal < 0.0, 0.0, v)


def _electron_loss(p, bg, ric):
    n_gas, b, divv = bg[0][:, None], bg[2][:, None], bg[3][:, None]
    p = p[None, :]
    br = b * 1.0e6 / 3.2
    beta2 = p * p / (1.0 + p * p)
    return (4.8e-4 * p * p * br * br * 9.11e-28 * 3.0e10 * GYR + ric[None, :] +
            3.05e-29 * n_gas * (1.0 + np.log(p / n_gas) / 74.8) / (ME * GEV) * C_LIGHT * GYR / beta2 + divv * p / 3.0)


def _nsub(pe, pp, bg, ric, dt):
    le = _electron_loss(pe[[0, -1]], bg, ric[[0, -1]])
    t = [np.abs(pe[0] / le[:, 0]), np.abs(pe[-1] / le[:, 1])]
    with np.errstate(divide="ignore"):
        t += [np.abs(pp[k] / (_coulomb_p(bg[0], pp[k], bg[1]) + bg[3] * pp[k] / 3.0)) for k in (0, -1)]
    target = np.minimum(dt / 10.0, 0.5 * np.minimum.reduce(t))
    e10 = np.floor(np.log10(target))
    ladder = np.array([1.0, 1.25, 1.6, 2.0, 2.5, 3.2, 4.0, 5.0, 6.4, 8.0])
    scale = np.array([10.0 ** int(e) for e in e10])
    used = ladder[np.maximum(0, np.searchsorted(ladder, target / scale, side="right") - 1)] * scale
    return np.maximum(10, np.ceil(dt / used)).astype(np.int64)


def _diffusion(case, p, bg):
    """D_pp rows: p^2 e^(-1/p) / (4 t_acc), or the floor p^2 / 4e5."""
    floor = np.broadcast_to((p * p / 4.0e5)[None, :], (bg.shape[1], len(p)))
    if case["dpp"] == 3:
        return floor
    length, dv, cs, beta = bg[4] * 3.0857e24, bg[5], bg[6], bg[7]
    mach = np.minimum(dv / cs, 0.5)
    if case["dpp"] == 1:
        t = math.sqrt(6.0 / 5.0) / 12.0 * (C_LIGHT / cs / cs) * length / np.sqrt(beta) / mach ** 3 * 0.125 / GYR
    else:
        x = cs / C_LIGHT
        theta = x ** 4 / 4.0 + x * x - (1.0 + 2.0 * x * x) * np.log(x) - 1.25
        t = 2.5e-3 / (x * theta) / (mach / 0.5) ** 4 * (length / (300.0 * 3.0857e21)) / (cs / 1500.0e5)
    d = (p * p * np.exp(-1.0 / p))[None, :] / (4.0 * t)[:, None]
    return np.where(((dv > 0.0) & (mach > 0.0))[:, None], d, floor)


def _cc_inverse(p, dp, loss, d, dt, dev):
    """Inverse of the Chang-Cooper matrix of every tracer, [tracer, n, n]."""
    t = [torch.from_numpy(np.ascontiguousarray(v)).to(dev) for v in (p, dp, loss, d, dt)]
    p, dp, loss, d, dt = t
    n = p.numel()
    bj = loss - 2.0 / p * d
    h = p[1:] - p[:-1]
    cf = 0.5 * (d[:, 1:] + d[:, :-1])
    w = 0.5 * (bj[:, 1:] + bj[:, :-1]) / cf * h
    aw = w.abs()
    small = aw < 0.1
    w2 = w * w
    big = torch.where(small, torch.exp(0.5 * aw) / (1.0 + w2 / 24.0 + w2 * w2 / 1920.0),
                      aw / -torch.expm1(-torch.where(small, torch.ones_like(aw), aw)))
    low = big * torch.exp(-aw)
    wp, wm = torch.where(w > 0, big, low), torch.where(w > 0, low, big)
    fh = cf / h
    t1 = dt[:, None] / dp
    z = torch.zeros_like(t1[:, :1])
    a = t1 * torch.cat([z, fh * wm], 1)
    c = t1 * torch.cat([fh * wp, z], 1)
    b = 1.0 + t1 * (torch.cat([z, fh * wp], 1) + torch.cat([fh * wm, z], 1))
    x = torch.eye(n, dtype=torch.float64, device=dev).expand(len(dt), n, n).clone()
    g = torch.empty_like(b)
    prev = None
    for j in range(n):
        den = b[:, j] - (a[:, j] * prev if j else 0.0)
        prev = c[:, j] / den
        g[:, j] = prev
        x[:, j] = (x[:, j] + (a[:, j, None] * x[:, j - 1] if j else 0.0)) / den[:, None]
    for j in range(n - 2, -1, -1):
        x[:, j] += g[:, j, None] * x[:, j + 1]
    return x


def _batch_exact(case, seed):
    """Electron runs on small grids: each segment of equal coefficients is a
    power of its inverse Chang-Cooper matrix (all entries non-negative, so
    the products lose no accuracy)."""
    w = _workload(case, seed)
    n, nt = case["n"], case["ntr"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    (pe, dpe), pp = _axis(n, 0.0, 6.0), _axis(n, -1.0, 8.0)[0]
    rows = [_ic_row(pe, float(z)) for z in w.z[:w.nsnap]]
    x = torch.from_numpy(w.cre0.reshape(nt, n).copy()).to(dev)
    for s in range(w.nsnap):
        ahead = s + 1 < w.nsnap
        cur, nxt = w.bg[s], w.bg[s + 1 if ahead else s]
        ns = _nsub(pe, pp, cur, rows[s], float(w.dt_snap[s]))
        nseg = np.ones(nt, dtype=np.int64)
        while ahead and (m := (nseg * 2 <= 16) & (nseg * 2 <= ns // 4)).any():
            nseg[m] *= 2
        for k in range(int(nseg.max())):
            for lo in range(0, nt, 512):
                idx = lo + np.flatnonzero(nseg[lo:lo + 512] > k)
                if not len(idx):
                    continue
                g = nseg[idx]
                steps = ((k + 1) * ns[idx]) // g - (k * ns[idx]) // g
                al = np.where(g > 1, (k + 0.5) / g, 0.0)
                bg = cur[:, idx] + al * (nxt[:, idx] - cur[:, idx])
                ric = rows[s][None, :] + al[:, None] * (rows[s + 1 if ahead else s] - rows[s])[None, :]
                loss = _electron_loss(pe, bg, np.zeros(n)) + ric
                m = _cc_inverse(pe, dpe, loss, _diffusion(case, pe, bg), w.dt_snap[s] / ns[idx], dev)
                at = torch.from_numpy(idx).to(dev)
                v, left = x[at].unsqueeze(2), torch.from_numpy(steps).to(dev)
                while int(left.max()) > 0:
                    v = torch.where((left % 2 == 1)[:, None, None], torch.bmm(m, v), v)
                    left = left // 2
                    if int(left.max()) > 0:
                        m = torch.bmm(m, m)
                x[at] = v.squeeze(2)
    return {"cre": x.cpu().numpy()}


def _synch_exact(case, seed):
    e = _emission_inputs(case, seed)
    n, nb, planes = case["n"], case["nbins"], case["planes"]
    tab = _synch_table(n, nb, planes)
    dp = _axis(n, 0.0, 6.0)[1]
    u = (np.log10(e["b"] / 1.0e-6) - LOGB[0]) * (planes / LOGB[1])
    ib = np.clip(np.floor(u).astype(int), 0, planes - 2)
    t = np.clip(u - ib, 0.0, 1.0)
    # bins from 2 on, up to the last whose successor is populated
    live = np.logical_and.accumulate(e["spec"][:, 3:] > 0.0, axis=1)
    wgt = np.where(live, e["spec"][:, 2:-1] * dp[2:-1], 0.0)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    tab, wgt, t = [torch.from_numpy(np.ascontiguousarray(v)).to(dev) for v in (tab[:, :, 2:-1], wgt, t)]
    lt = torch.log(tab)
    ib = torch.from_numpy(ib).to(dev)
    out = np.empty((case["ntr"], nb))
    for i in range(0, case["ntr"], 256):
        j, f = ib[i:i + 256], t[i:i + 256, None, None]
        k0, k1 = tab[j], tab[j + 1]
        k = torch.where((k0 > 0.0) & (k1 > 0.0), torch.exp((1.0 - f) * lt[j] + f * lt[j + 1]), (1.0 - f) * k0 + f * k1)
        out[i:i + 256] = (k * wgt[i:i + 256, None, :]).sum(2).cpu().numpy()
    amp = math.sqrt(3.0) * 4.8e-10 ** 3 * e["b"] / (2.0 * 9.11e-28 * C_LIGHT * C_LIGHT) / (4.0 * math.pi)
    return amp[:, None] * out


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        if case["species"] != 1 or case["fp32"] or case["ntr"] * case["nsnap"] * case["n"] ** 3 > 3e10:
            return None
        return _batch_exact(case, seed)
    if kind == "solve":
        a, b, c, q, x = [t.numpy() for t in _solve_systems(case, seed, "cpu")]
        n = case["nrow"]
        x = SOLVE_DT * q + x
        g = np.zeros_like(x)
        for j in range(n):
            den = b[:, j] - (a[:, j] * g[:, j - 1] if j else 0.0)
            g[:, j] = c[:, j] / den
            x[:, j] = (x[:, j] + (a[:, j] * x[:, j - 1] if j else 0.0)) / den
        for j in range(n - 2, -1, -1):
            x[:, j] += g[:, j] * x[:, j + 1]
        return x
    if kind == "ic":
        e = _emission_inputs(case, seed)
        tab = _ic_table(case["n"], case["nbins"], e["z"])
        return {"table": tab, "eps": e["spec"] @ (tab * _axis(case["n"], 0.0, 6.0)[1]).T}
    if kind == "had":
        e = _emission_inputs(case, seed)
        p, dp = _axis(case["n"], -1.0, 8.0)
        tw = np.concatenate([[0.0], dp[1:]]) + np.concatenate([dp[1:], [0.0]])
        energy = 10.0 ** (-1.0 + 6.0 / case["nbins"] * np.arange(case["nbins"]))
        km = energy[:, None] * 0.5 * (p / np.sqrt(1.0 + p * p) * tw)[None, :] * e["fk"]
        return e["n_gas"][:, None] * (e["spec"] @ km.T)
    if kind == "synch":
        return _synch_exact(case, seed)
    return None
