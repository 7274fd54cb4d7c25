"""Lane-group batched solve against the one-thread Thomas sweep, bit for bit.

Systems of up to 1,024 rows run on lane groups, longer ones on one thread
each.  Each system here is solved as it is and again with identity rows
that make it 1,100 rows long, which sends it down the one-thread path; its own
rows must come out identical, whatever the signs and the dominance, also
where a system holds infinities or NaN, in its last row among others (and its
neighbours in the wave stay untouched).  Those systems take the identity rows
before their own: rows appended would bring 0 x infinity into the last one."""
import numpy as np
import pytest

import croma_hip as ch

pytestmark = pytest.mark.gpu

LONG = 1100
ROWS = [1, 2, 3, 7, 8, 9, 16, 17, 31, 33, 64, 65, 127, 129, 200, 256, 257, 511, 512, 513, 700, 1024]


def _systems(kind, ns, nr, rng):
    if kind == "cc":  # Chang-Cooper: non-negative couplings, dominant diagonal
        a = rng.uniform(0.0, 2.0, (ns, nr)) * 10.0 ** rng.uniform(-3, 3, (ns, 1))
        c = rng.uniform(0.0, 2.0, (ns, nr)) * 10.0 ** rng.uniform(-3, 3, (ns, 1))
        b = 1.0 + rng.uniform(0.0, 0.1, (ns, nr)) + a + c
        x = 10.0 ** rng.uniform(-30, 5, (ns, nr))
    else:  # any signs, no dominance
        a, c, x = (rng.normal(size=(ns, nr)) for _ in range(3))
        b = rng.normal(size=(ns, nr)) + np.where(rng.random((ns, nr)) < 0.5, 3.0, -0.5)
        if kind == "special":
            for v in (np.inf, -np.inf, np.nan, 1e300, -0.0):
                for arr in (a, c, x):
                    arr[rng.integers(ns), rng.integers(nr)] = v
            x[ns // 2] = rng.normal(size=nr)
            a[ns // 2], c[ns // 2] = rng.normal(size=(2, nr))
            x[ns // 2, -1] = np.inf  # the last row alone: the rows before it follow from it
    q = 10.0 ** rng.uniform(-6, 0, (ns, nr))
    a[:, 0] = rng.normal(size=ns)   # ignored by the sweep
    c[:, -1] = rng.normal(size=ns)  # ignored by the sweep
    return a, b, c, q, x


def _long(v, pad, nr, before=False):
    out = np.full((v.shape[0], LONG), pad)
    if before:
        out[:, LONG - nr:] = v
    else:
        out[:, :nr] = v
    return out


@pytest.mark.parametrize("kind", ["cc", "general", "special"])
def test_lane_groups_equal_the_one_thread_sweep(kind):
    rng = np.random.default_rng(7)
    dt = 0.0137
    for nr in ROWS:
        for ns in (1, 5, 67):
            a, b, c, q, x = _systems(kind, ns, nr, rng)
            print(f"[solve] {kind} {ns} x {nr}", flush=True)
            got, _ = ch.solve_cc_batch(a, b, c, q, x, dt)
            c0, a0, before = c.copy(), a.copy(), kind == "special"
            if before:
                a0[:, 0] = -0.0  # the row before comes out as 0: -0 x 0 changes no sum
            else:
                c0[:, -1] = 0.0
            want, _ = ch.solve_cc_batch(_long(a0, 0.0, nr, before), _long(b, 1.0, nr, before),
                                        _long(c0, 0.0, nr, before), _long(q, 0.0, nr, before),
                                        _long(x, 0.0, nr, before), dt)
            want = want[:, LONG - nr:] if before else want[:, :nr]
            if kind == "special":
                number = ~np.isnan(want)
                assert np.isinf(want[ns // 2, -1]) and number.any()
                assert np.array_equal(got, want, equal_nan=True), (nr, ns, np.argwhere(got != want)[:3])
                assert np.array_equal(np.signbit(got)[number], np.signbit(want)[number]), (nr, ns)
            else:
                assert np.array_equal(got, want), (nr, ns, np.argwhere(got != want)[:3])
