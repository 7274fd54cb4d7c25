"""The C host runtime on a stand-in for the device layer (device_stub.c, host
memory, kernels that compute nothing and are recorded): which launches a call
takes, what it reserves and what it does when a reservation fails.  No GPU."""
import ctypes as C
import glob
import os
import subprocess
import threading
import time

import numpy as np
import pytest

import croma_hip as ch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "croma-fp_amd")


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libcroma_stub.so")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-O1", "-std=gnu11", "-ffp-contract=off", "-pthread", "-w",
                           "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(REPO, "include"), "-o", out,
                           *sorted(glob.glob(os.path.join(PKG, "host", "*.c"))),
                           os.path.join(REPO, "tests", "device_stub.c"), "-lm"])
    return out


@pytest.fixture
def stub(stub_path, monkeypatch):
    monkeypatch.setattr(ch, "LIB_PATH", stub_path)
    monkeypatch.setattr(ch, "_lib", None)
    L = ch.lib()
    L.stub_peak.restype = L.stub_live.restype = C.c_size_t
    L.stub_set_limit.argtypes = [C.c_size_t, C.c_size_t]
    L.stub_fix_next.argtypes = [C.c_size_t]
    L.stub_set_cost.argtypes = [C.c_int, C.c_double, C.c_double]
    L.stub_set_host_alloc_hook.argtypes = [C.c_void_p]
    L.ck_set_device(0)
    L.stub_reset()
    yield L
    L.ck_set_device(0)


def _launches(L):
    m, r, t = ((C.c_int * 4096)() for _ in range(3))
    k = L.stub_launches(m, r, t, 4096)
    return [(m[i], r[i], t[i]) for i in range(k)]


def _snapshot(ctx, nt, nsub):
    n = ctx.n
    bg = np.ones((8, nt))
    row = np.ones(n)
    fqe = np.zeros((n, n))
    fqe[n // 2:] = 1.0
    x = np.ones(nt * n)
    zero = np.zeros(nt * n)
    crp, cre = x.copy(), x.copy()
    nsub = np.asarray(nsub, np.int32)
    ctx.execute_snapshot(nsub, nsub, True, 0.0, 0.01, bg, row, 1.0, 1.0, bg, row, 1.0, 1.0, zero, zero, fqe.ravel(),
                         np.full(n, n // 2, np.int32), np.ones(nt), None, crp, cre)
    return crp, cre


# tracers, substeps, most segments: the rows that the calls' own substep
# counts ask for, not tracers x most segments
@pytest.mark.parametrize("nt,nsub,segs", [(500, 4, 16), (300, 37, 4096), (64, 4096, 1024)])
def test_drop_in_reserves_the_rows_it_writes(stub, nt, nsub, segs):
    n = 64
    ctx = ch.Context(n, ch.default_params(coeff_interp_max_segments=segs, coeff_interp_min_steps=4))
    try:
        _snapshot(ctx, nt, np.full(nt, nsub))
        assert [m for m, _, _ in _launches(stub)] == [2, 3]  # the split launch
        most = 1
        while most * 2 <= min(segs, nsub // 4):
            most *= 2
        rows = nt * most
        # two arrays of rows, rounded up by at most 1/32 and 256 rows; the state,
        # sources and backgrounds are below 8 arrays of the spectra and the weights
        other = 8 * nt * n * 8 + 4 * n * n * 8 + (1 << 20)
        assert stub.stub_peak() <= 2 * (rows * (1 + 1 / 32) + 256) * n * 8 + other
    finally:
        ctx.close()


@pytest.mark.parametrize("fp32", [False, True])
def test_drop_in_without_room_for_the_rows_runs_the_in_kernel_contraction(stub, fp32):
    n, nt = 128, 400
    ctx = ch.Context(n, ch.default_params(coeff_interp_max_segments=1024, coeff_interp_min_steps=1))
    try:
        ctx.set_coeff_precision(fp32)
        state = nt * n * 8
        for largest, free in ((4 * state, 1 << 38), (1 << 40, 100 * state)):
            stub.stub_reset()
            stub.stub_set_limit(largest, free)
            before = stub.stub_live()
            crp, cre = _snapshot(ctx, nt, np.full(nt, 1024))  # 1024 segments: 2048 x state
            modes = [m & ~4 if fp32 else m for m, _, _ in _launches(stub)]
            assert modes == [1]
            assert np.all(crp == 1.0) and np.all(cre == 1.0)
            # nothing of a failed reservation is left
            assert stub.stub_live() - before < 12 * state + (4 << 20)
        # fewer segments: room again
        stub.stub_reset()
        stub.stub_set_limit(1 << 40, 1 << 38)
        _snapshot(ctx, nt, np.full(nt, 16))
        assert [m & ~4 if fp32 else m for m, _, _ in _launches(stub)] == [2, 3]
    finally:
        ctx.close()


def _made(L, d):
    out = (C.c_int * 3)()
    L.stub_made(d, out)
    return list(out)


def _in_new_thread(L, fn):
    """fn in a thread that has chosen no device; its device afterwards."""
    out = {}

    def run():
        try:
            out["value"] = fn()
        except Exception as e:  # pragma: no cover
            out["error"] = e
        out["device"] = L.ck_get_device()

    t = threading.Thread(target=run)
    t.start()
    t.join()
    assert "error" not in out, out["error"]
    assert out["device"] == 0
    return out["value"]


@pytest.mark.parametrize("first", ["own", "thread"])
def test_calls_from_another_threads_device(stub, first):
    """A context of device 3 used by a thread whose device is 0: transfers and
    the emission calls make what they need on device 3 and leave the thread's
    device as it was."""
    stub.ck_set_device(3)
    n, nt, nb = 64, 9000, 8  # 4.6 MB: through the pinned ring
    ctx = ch.Context(n, ch.default_params())
    b = ch.Batch(ctx, nt, ch.SPECIES_ELECTRON, 1)
    x = np.random.default_rng(1).uniform(size=nt * n)
    fic = np.ones(nb * n)
    table = np.ones(200 * 16 * n)

    def transfer():
        b.set_state(None, x)
        return np.array_equal(b.get_state()[1], x)

    def emission():
        ctx.emission_ic(x, fic, nb, ch.EMIS_FP64)
        ctx.emission_kernel_table(ch.TABLE_IC, nb, 8.0, 20.0, 0.1)
        p = ch.SynchPlan(ctx, table, 16, 200, -8.0, 100.0)
        p.run(x, np.full(nt, 1e-6))
        p.run(np.tile(x, 2), np.full(2 * nt, 1e-6))
        p.close()
        return True

    try:
        stub.stub_reset()
        if first == "own":
            assert transfer() and emission()
        assert _in_new_thread(stub, transfer) and _in_new_thread(stub, emission)
        assert transfer() and emission()
        assert _made(stub, 0) == [0, 0, 0]
        assert _made(stub, 3)[0] >= 4  # the ring's streams
    finally:
        b.close()
        ctx.close()


def test_ic_end_rates_of_many_redshifts(stub):
    """The nsub estimate's IC rates at the first and last bin, batched and
    cached: the row's own values bit for bit, in the order asked for, over more
    redshifts than the cache holds, with repeats; also for a redshift that is
    not a number (equal to none in the cache)."""
    ctx = ch.Context(64, ch.default_params())
    try:
        stub.ch_ctx_ic_ends.argtypes = [C.c_void_p, C.c_int, C.POINTER(C.c_double), C.POINTER(C.c_double)]
        stub.ch_ctx_ic_ends.restype = None
        dp = C.POINTER(C.c_double)

        def ends(z):
            z = np.ascontiguousarray(z, np.float64)
            out = np.full((len(z), 2), 12345.0)
            stub.ch_ctx_ic_ends(C.c_void_p(ctx.h), len(z), z.ctypes.data_as(dp), out.ctypes.data_as(dp))
            return out

        few = np.array([0.0, 0.3, 0.1, 0.3, 6.0])
        want = np.array([[ctx.ic_cooling_row(v)[0][i] for i in (0, -1)] for v in few])
        assert np.array_equal(ends(few), want) and np.array_equal(ends(few), want)
        many = np.linspace(0.0, 2.0, 700)
        got = ends(many)
        assert np.array_equal(got[::-1], ends(many[::-1])) and np.array_equal(ends(few), want)
        assert np.array_equal(got[350], [ctx.ic_cooling_row(many[350])[0][i] for i in (0, -1)])
        got, row = ends([0.1, np.nan, 0.3]), ctx.ic_cooling_row(np.nan)[0]
        assert np.array_equal(got[[0, 2]], want[[2, 1]])
        assert np.array_equal(got[1], row[[0, -1]], equal_nan=True)
    finally:
        ctx.close()


def test_cancel_while_a_launch_is_put_together(stub):
    """A request cancelled after the scheduler has counted it for a launch (the
    growing task list's allocation is such a moment) still comes to an end."""
    def chunk(nt, nsnap):
        return srv.submit(64, ch.SPECIES_ELECTRON, 1, 0.01 * np.arange(nsnap + 1)[::-1], np.full(nsnap, 0.01),
                          np.ones((nsnap + 1, 8, nt)), cre=np.ones(nt * 64))

    srv = ch.Server(64 << 20)
    me, ids, hits = threading.get_ident(), [], []

    @C.CFUNCTYPE(None)
    def hook():  # the submitting thread allocates too
        if threading.get_ident() != me and not hits:
            hits.append(1)
            srv.cancel(ids[0])

    try:
        srv.wait(chunk(4, 1))  # the class's first, small task list
        ids.append(2)          # the next request's number
        stub.stub_set_host_alloc_hook(C.cast(hook, C.c_void_p))
        assert chunk(500, 50) == ids[0]
        end = time.time() + 5.0
        while srv.poll(ids[0]) == 0 and time.time() < end:
            time.sleep(0.01)
        assert hits and srv.poll(ids[0]) == ch.ECANCELED
        assert srv.stats()["in_use_bytes"] == 0
    finally:
        stub.stub_set_host_alloc_hook(None)
        srv.close()


def test_server_works_on_the_device_it_was_made_on(stub):
    stub.ck_set_device(5)
    srv = ch.Server(64 << 20)
    try:
        stub.stub_reset()
        rid = srv.submit(64, ch.SPECIES_ELECTRON, 1, np.array([0.01, 0.0]), np.array([0.01]), np.ones((2, 8, 30)),
                         cre=np.ones(30 * 64))
        assert np.all(srv.wait(rid)[1] == 1.0)
        assert _made(stub, 0) == [0, 0, 0] and _made(stub, 5)[2] > 0
    finally:
        srv.close()


def test_get_tile_tells_what_a_run_took(stub):
    def run(ctx, species, nt, ns):
        b = ch.Batch(ctx, nt, species, ns)
        for s in range(ns):
            b.set_background(s, np.ones((8, nt)))
        b.set_state(None, np.ones(nt * ctx.n))
        stub.stub_reset()
        b.run(0, ns, ns, np.linspace(0.1, 0.0, ns + 1), np.full(ns, 0.01))
        b.close()
        return ctx.get_tile(species != ch.SPECIES_ELECTRON), _launches(stub)

    ctx = ch.Context(128, ch.default_params())
    try:
        e, p = ctx.get_tile(False), ctx.get_tile(True)
        tile, log = run(ctx, ch.SPECIES_ELECTRON, 100, 5)
        assert tile[2:] == (5, 0) and [(r, t) for _, r, t in log] == [(tile[0], 100)]  # one window
        assert ctx.get_tile(True) == p
        tile, log = run(ctx, ch.SPECIES_ELECTRON, 70000, 2)
        assert tile[2] == 1 and len(log) == 2 and log[0][1] == tile[0] != 4
        tile, log = run(ctx, ch.SPECIES_ELECTRON_PROTON, 100, 3)
        assert tile[2:] == (1, 1) and [m for m, _, _ in log] == [2, 3] * 3
        _snapshot(ctx, 50, np.full(50, 8))
        assert ctx.get_tile(True)[3] == 1
        ctx.set_tile(8, 2, 1, protons=0, secondary_gemm=0)
        assert ctx.get_tile(False) == (8, 2, 1, 0) and e[3] == 0
    finally:
        ctx.close()
    ctx = ch.Context(128, ch.default_params(dpp_model=1, eta_dpp_cap=0.1))
    try:
        tile, log = run(ctx, ch.SPECIES_ELECTRON_PROTON, 100, 3)
        assert tile[2:] == (3, 0) and [m for m, _, _ in log] == [1]
    finally:
        ctx.close()


def test_tuned_runs_keep_the_windows_by_size(stub):
    """An autotuner times rows, waves and the contraction; the snapshots of a
    window stay a matter of size, and a tile that wins one snapshot at a time
    does not displace the rule's where runs are slower with it."""
    n, nt, ns = 128, 100, 6
    z, dt = np.linspace(0.1, 0.0, ns + 1), np.full(ns, 0.01)
    for costs, rows in (({4: (1.5, 0.1), 8: (2.0, 0.1), 16: (0.0, 1.0)}, 4),   # 16 rows win one snapshot alone
                        ({4: (2.0, 0.5), 8: (2.0, 0.1), 16: (0.5, 0.3)}, 16)):  # and here runs too
        ctx = ch.Context(n, ch.default_params())
        ctx.set_graphs(False)  # every launch on the record
        b = ch.Batch(ctx, nt, ch.SPECIES_ELECTRON, ns)
        try:
            for s in range(ns):
                b.set_background(s, np.ones((8, nt)))
            b.set_state(None, np.ones(nt * n))
            for r, c in costs.items():
                stub.stub_set_cost(r, *c)
            tile = b.autotune(0, ns, z, dt)
            assert tile[0] == rows and tile == ctx.get_tile(False)
            stub.stub_reset()
            b.run(0, ns, ns, z, dt)
            assert [(r, t) for _, r, t in _launches(stub)] == [(rows, nt)]  # one window
            assert ctx.get_tile(False) == (rows, tile[1], ns, 0)
            ctx.set_tile(8, 2, 1, protons=0)
            stub.stub_reset()
            b.run(0, ns, ns, z, dt)
            assert [r for _, r, _ in _launches(stub)] == [8] * ns  # as set
        finally:
            b.close()
            ctx.close()
    ctx = ch.Context(n, ch.default_params())
    try:
        ctx.autotune(False, 64)
        b = ch.Batch(ctx, nt, ch.SPECIES_ELECTRON, ns)
        for s in range(ns):
            b.set_background(s, np.ones((8, nt)))
        b.set_state(None, np.ones(nt * n))
        stub.stub_reset()
        b.run(0, ns, ns, z, dt)
        b.close()
        assert len(_launches(stub)) == 1
    finally:
        ctx.close()


@pytest.mark.parametrize("pipelined", [False, True])
def test_graphs_do_not_outlive_the_segment_rows(stub, pipelined):
    """Growing the segment rows replaces both arrays; a window whose launch key
    repeats (the first array back at its old address, the same row count) must
    not replay a graph that writes to the second one's old address."""
    n, nt, ns = 64, 40, 6
    z, dt = np.linspace(0.06, 0.0, ns + 1), np.full(ns, 0.01)
    ctx = ch.Context(n, ch.default_params(coeff_interp_max_segments=1))
    ctx.set_nsub_device(False)
    ctx.set_pipeline(pipelined)
    b = ch.Batch(ctx, nt, ch.SPECIES_ELECTRON_PROTON, ns)
    try:
        for s in range(ns):
            b.set_background(s, np.ones((8, nt)))
        b.set_state(np.ones(nt * n), np.ones(nt * n))
        stub.stub_fix_next(256 * n * 8)  # rows in steps of 256
        assert b.run(0, ns, ns, z, dt).graph_launches > 0
        # more segments allowed, none taken: the same row counts
        ctx.set_params(ch.default_params(coeff_interp_max_segments=64, coeff_interp_min_steps=1 << 20))
        stub.stub_fix_next(nt * 64 * n * 8)
        b.run(0, ns, ns, z, dt)
    finally:
        b.close()
        ctx.close()


def test_drop_in_graph_does_not_outlive_its_batch(stub):
    """A call of another shape that fails after the old batch is gone leaves no
    graph of that batch for the next call of the old shape."""
    n, nt = 64, 40
    ctx = ch.Context(n, ch.default_params())
    try:
        for failing in (True, False):
            stub.stub_fix_next(256 * n * 8)
            for _ in range(4):  # eager, captured, replayed
                _snapshot(ctx, nt, np.full(nt, 4))
            if failing:
                stub.stub_set_limit(1 << 10, 1 << 38)
                with pytest.raises(ch.CromaHipError):
                    _snapshot(ctx, 2 * nt, np.full(2 * nt, 4))
                stub.stub_set_limit(1 << 40, 1 << 38)
    finally:
        ctx.close()
