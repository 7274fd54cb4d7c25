"""Transfers through the pinned ring: arrays on both sides of its size and
piece lines come back unchanged, from several threads at once on one context
(one has the ring and the context's work memory, the others their own), and
emission calls of changing sizes reuse the context's memory without a trace of
the call before."""
import threading

import numpy as np
import pytest

import croma_hip as ch

pytestmark = pytest.mark.gpu


def _round_trip(ctx, nt, seed, out, key):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.0, 1.0, nt * ctx.n)
    y = rng.uniform(0.0, 1.0, nt * ctx.n)
    b = ch.Batch(ctx, nt, ch.SPECIES_ELECTRON_PROTON, 1)
    try:
        b.set_state(y, x)
        crp, cre = b.get_state()
    finally:
        b.close()
    out[key] = np.array_equal(cre, x) and np.array_equal(crp, y)


# 64 bins x 8 bytes: 4 MiB at 8,192 tracers, 1 MiB pieces
@pytest.mark.parametrize("nt", [1, 8191, 8192, 8193, 10240, 16385, 40961])
def test_state_round_trip(nt):
    ctx = ch.Context(64, ch.default_params())
    out = {}
    try:
        _round_trip(ctx, nt, nt, out, 0)
    finally:
        ctx.close()
    assert out[0]


def test_threads_share_the_ring():
    ctxs = [ch.Context(64, ch.default_params()) for _ in range(3)]
    out = {}
    try:
        for rep in range(3):
            th = [threading.Thread(target=_round_trip, args=(c, 20000 + 7 * i, 10 * rep + i, out, (rep, i)))
                  for i, c in enumerate(ctxs)]
            for t in th:
                t.start()
            for t in th:
                t.join()
    finally:
        for c in ctxs:
            c.close()
    assert len(out) == 9 and all(out.values())


def test_emission_work_memory_across_sizes_and_threads():
    n, nb = 64, 40
    rng = np.random.default_rng(3)
    ctx = ch.Context(n, ch.default_params())
    fic = rng.uniform(0.1, 1.0, (nb, n))
    dp = ctx.grid(1)[1]
    errs = []

    def one(nt, seed):
        x = np.random.default_rng(seed).uniform(0.0, 1.0, (nt, n))
        eps, _ = ctx.emission_ic(x, fic.ravel(), nb, ch.EMIS_FP64)
        want = x @ (fic * dp).T
        errs.append(float(np.max(np.abs(eps - want) / want)))

    try:
        for nt in (30000, 17, 9000, 30001):
            one(nt, nt)
        th = [threading.Thread(target=one, args=(12000 + i, i)) for i in range(4)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    finally:
        ctx.close()
    assert len(errs) == 8 and max(errs) < 1e-12  # the FP64 mode's bar: 64 positive terms
