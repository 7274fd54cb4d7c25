"""Segment bookkeeping of the fused kernel against the CPU oracle: segment
counts below, at and above the number whose scalars the lanes evaluate at a
time, the direct-t_acc switch and the eta cap (both per-segment scalars), and
rows without diffusion (E_max so low that the protons' D_pp underflows to
zero), in every launch mode.  Tolerance of the main parity test."""
import numpy as np
import pytest

import croma_hip as ch
import run_oracle
from workloads import hip_params, rel_err, run_hip, small_workload

pytestmark = pytest.mark.gpu

CASES = [
    # n, rows per lane, ntracer, species, dpp, split, params
    (64, 16, 21, 1, 2, 0, {"coeff_interp_max_segments": 64, "coeff_interp_min_steps": 1}),
    (64, 4, 13, 3, 1, 0, {"coeff_interp_max_segments": 5, "coeff_interp_min_steps": 1}),
    (128, 8, 19, 3, 2, 1, {"coeff_interp_max_segments": 64, "coeff_interp_min_steps": 2}),
    (256, 8, 9, 3, 1, 1, {"coeff_interp_max_segments": 1}),
    (512, 16, 7, 1, 2, 0, {"coeff_interp_max_segments": 33, "coeff_interp_min_steps": 1}),
    (64, 4, 11, 3, 4, 0, {"t_acc_direct_gyr": 0.2, "t_acc_off_gyr": 1.5, "t_off_gyr": 0.06}),
    (128, 4, 15, 3, 2, 0, {"eta_dpp_cap": 0.05, "reacc_window_mode": 1}),
    (128, 16, 15, 3, 1, 1, {"epmax": 1.0e3}),
    (128, 16, 15, 2, 1, 0, {"epmax": 1.0e3}),
]


@pytest.mark.parametrize("case", CASES, ids=[f"n{c[0]}-r{c[1]}-sp{c[3]}-dpp{c[4]}-{'-'.join(c[6])}" for c in CASES])
def test_segments_match_oracle(case):
    n, r, nt, sp, dpp, split, extra = case
    w = small_workload(n, nt, 2, sp, dpp, seed=23)
    crp_ref, cre_ref = run_oracle.run_workload(w, run_oracle.oracle_params(w, **extra))
    ctx = ch.Context(n, hip_params(w, **extra))
    try:
        for occ in (1, 2):
            ctx.set_tile(r, occ, 1, secondary_gemm=split)
            crp, cre, _ = run_hip(w, ctx)
            for name, got, want in (("electrons", cre, cre_ref), ("protons", crp, crp_ref)):
                err, ok = rel_err(got, want)
                print(f"[segments] n={n} r={r} occ={occ} {name} max rel err {err:.3e}", flush=True)
                assert ok, (name, occ, err)
    finally:
        ctx.close()
    assert np.all(np.isfinite(cre))


@pytest.mark.parametrize("n,species", [(64, 1), (128, 3), (256, 3), (512, 1)])
@pytest.mark.parametrize("fp32", [False, True])
def test_uninterpolated_segments_ignore_the_next_row(n, species, fp32):
    """Drop-in calls without interpolation, by the flag or because every tracer
    has one segment: the next IC row and backgrounds may hold anything."""
    w = small_workload(n, 21, 1, species, 1, seed=11)
    nt = w.ntracer
    crp0 = w.crp0 if w.protons else np.zeros(nt * n)
    zero = np.zeros(nt * n)
    for allow, extra in ((False, {}), (True, {"coeff_interp_max_segments": 1})):
        ctx = ch.Context(n, hip_params(w, **extra))
        try:
            ctx.set_coeff_precision(fp32)
            row, m1, p1 = ctx.ic_cooling_row(float(w.z[0]))
            f = w.bg[0]
            ns, non = ctx.nsub(float(w.dt_snap[0]), f[0], f[1], f[2], f[3], row[0], row[-1], f[4], f[5])
            fqe, npmin = ctx.secondary_weights()
            out = []
            for nxt in (1.0, np.inf, -np.inf, np.nan):
                crp, cre = crp0.copy(), w.cre0.copy()
                ctx.execute_snapshot(ns, non, allow, 0.0, float(w.dt_snap[0]), f, row, m1, p1,
                                     np.full((8, nt), nxt), np.full(n, nxt), nxt, nxt, zero, zero, fqe.ravel(), npmin,
                                     w.mass, None, crp, cre)
                out.append((crp, cre))
        finally:
            ctx.close()
        assert np.all(np.isfinite(out[0][1]))
        for crp, cre in out[1:]:
            assert np.array_equal(cre, out[0][1]) and np.array_equal(crp, out[0][0])
