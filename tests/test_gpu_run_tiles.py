"""Launch rules by size (no tile set): on both sides of each line, a run over
several snapshots in one window equals the same snapshots run one at a time
bit for bit, and a run at a fixed tile to rounding; the drop-in's split launch
equals the in-kernel contraction that weights below the first proton row ask
for."""
import ctypes as C

import numpy as np
import pytest

import croma_hip as ch
import synth
from workloads import hip_params, run_hip, small_workload

pytestmark = pytest.mark.gpu

CASES = [
    # n, ntracer, species, D_pp, snapshots, fixed tile, params
    (64, 37, 1, 3, 5, (16, 1), {}),
    (64, 16384, 1, 1, 2, (4, 2), {}),   # 2^20 rows
    (64, 16385, 1, 1, 2, (4, 2), {}),
    (128, 8193, 1, 2, 3, (16, 2), {}),
    (256, 300, 1, 2, 18, (16, 1), {}),  # two windows of the longest kind and a rest
    (256, 24577, 1, 2, 2, (8, 1), {}),  # above 6 * 2^20 rows
    (512, 40, 1, 2, 3, (8, 2), {}),
    (64, 50, 3, 1, 4, (8, 1), {}),
    (128, 700, 3, 2, 3, (8, 2), {}),
    (256, 60, 3, 1, 3, (16, 1), {}),
    (512, 30, 3, 2, 3, (8, 1), {}),
    (128, 90, 3, 2, 4, (4, 1), {"eta_dpp_cap": 0.1, "reacc_window_mode": 1}),
]


def _run(w, tile, one_by_one, extra):
    ctx = ch.Context(w.n, hip_params(w, **extra))
    try:
        if tile:
            ctx.set_tile(*tile)
        b = ch.Batch(ctx, w.ntracer, w.species, w.nsnap)
        b.set_state(w.crp0 if w.protons else None, w.cre0, mass=w.mass)
        for s in range(w.nsnap):
            b.set_background(s, w.bg[s])
        el = 0.0
        for s in range(w.nsnap) if one_by_one else [0]:
            b.run(s, s + 1 if one_by_one else w.nsnap, w.nsnap, w.z, w.dt_snap, elapsed=el)
            el += float(w.dt_snap[s])
        out = b.get_state()
        b.close()
        return out
    finally:
        ctx.close()


@pytest.mark.parametrize("case", CASES, ids=[f"n{c[0]}-{c[1]}-sp{c[2]}-{c[4]}" for c in CASES])
def test_windows_and_tiles_by_size(case):
    n, nt, sp, dpp, ns, tile, extra = case
    print(f"[run tiles] n={n} tracers={nt} species={sp}", flush=True)
    w = synth.make_workload(n=n, ntracer=nt, nsnap=ns, species=sp, dpp_model=dpp, seed=31, z0=0.005 * ns)
    whole, single, fixed = _run(w, None, False, extra), _run(w, None, True, extra), _run(w, tile, False, extra)
    for a, b, f in zip(whole, single, fixed):
        assert np.array_equal(a, b)
        m = np.abs(f) > 1e-30
        assert np.all(np.isfinite(a))
        # the solve's own rounding between launch shapes, far below the 1e-10 bar
        assert not m.any() or np.max(np.abs(a[m] - f[m]) / np.abs(f[m])) < 1e-11


@pytest.mark.parametrize("n", [64, 128, 256, 512])
def test_snapshot_split_equals_in_kernel_contraction(n):
    w = small_workload(n, 75, 1, 3, 1, seed=5)
    out = []
    for below in (False, True):
        ctx = ch.Context(n, hip_params(w))
        try:
            row, m1, p1 = ctx.ic_cooling_row(float(w.z[0]))
            f = w.bg[0]
            ns, non = ctx.nsub(float(w.dt_snap[0]), f[0], f[1], f[2], f[3], row[0], row[-1], f[4], f[5])
            fqe, npmin = ctx.secondary_weights()
            # first rows off a multiple of 16, so that the contraction starts below them
            npmin = np.maximum(npmin, npmin.min() // 16 * 16 + 5).astype(np.int32)
            fqe = np.where(np.arange(n)[:, None] < npmin.min(), 0.0, fqe.reshape(n, n))
            if below:
                fqe[npmin.min() - 1] = 1e-3  # the sums start above this row: it counts for nothing
            crp, cre = w.crp0.copy(), w.cre0.copy()
            zero = np.zeros(w.ntracer * n)
            for _ in range(4):  # eager, captured, replayed
                ctx.execute_snapshot(ns, non, True, 0.0, float(w.dt_snap[0]), w.bg[0], row, m1, p1, w.bg[1], row, m1,
                                     p1, zero, zero, fqe.ravel(), npmin, w.mass, None, crp, cre)
            assert ctx.get_tile(True)[3] == (0 if below else 1)  # the launch it took
            out.append((crp, cre))
        finally:
            ctx.close()
    for a, b in zip(*out):
        m = np.abs(b) > 1e-30
        assert np.max(np.abs(a[m] - b[m]) / np.abs(b[m])) < 1e-11


def test_snapshot_rows_follow_the_substep_counts():
    """Two species, as many segments allowed as a call could ask for: the rows
    reserved are those of the calls' own substep counts, and the result is that
    of a limit no tracer reaches."""
    n = 64
    w = small_workload(n, 75, 1, 3, 1, seed=5)
    out = []
    for segs in (4096, 1 << 24):  # 75 x 2^24 rows of 64 bins: 1.3e12 bytes
        ctx = ch.Context(n, hip_params(w, coeff_interp_max_segments=segs, coeff_interp_min_steps=2))
        try:
            row, m1, p1 = ctx.ic_cooling_row(float(w.z[0]))
            f = w.bg[0]
            ns, non = ctx.nsub(float(w.dt_snap[0]), f[0], f[1], f[2], f[3], row[0], row[-1], f[4], f[5])
            assert ns.max() // 2 < 4096
            fqe, npmin = ctx.secondary_weights()
            crp, cre = w.crp0.copy(), w.cre0.copy()
            zero = np.zeros(w.ntracer * n)
            ctx.execute_snapshot(ns, non, True, 0.0, float(w.dt_snap[0]), f, row, m1, p1, w.bg[1], row, m1, p1, zero,
                                 zero, fqe.ravel(), npmin, w.mass, None, crp, cre)
            out.append((crp, cre))
        finally:
            ctx.close()
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)


def test_failed_allocation_leaves_no_error_behind():
    """A refused allocation is reported by its own call, not by the check after
    the next launch (a call that does without what it could not get goes on)."""
    ck_malloc = ch.lib().ck_malloc
    ck_malloc.restype, ck_malloc.argtypes = C.c_void_p, [C.c_size_t]
    w = small_workload(64, 20, 1, 1, 1)
    ctx = ch.Context(64, hip_params(w))
    try:
        want = run_hip(w, ctx)[1]
        assert not ck_malloc(1 << 50)
        assert np.array_equal(run_hip(w, ctx)[1], want)
    finally:
        ctx.close()
