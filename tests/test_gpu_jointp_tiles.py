"""jointp at the edges of its tiles: genealogies around a stage (256 rows, 128
above 8 parameters), its quarters and chunks; points around the 16-point
tile and the wide workgroups; every number of parameters.

Values and effective sample numbers against the oracle (REF_COMPAT) and a
float64 numpy log-sum-exp (EXACT).  Bound: a term's sum has up to 33
products below 2^12 in size, so its rounding is below 33 * 2^12 * 2^-53 =
1.5e-11 absolute and moves log-sum-exp by no more.  The oracle's REF_COMPAT
terms come from eexp's degree-10 Taylor series on [0, ln 2), which falls
short by up to (ln 2)^11 / 11! = 4.5e-10 of a term (REF_TOL); the engine's
do not.  The same points are the same bits alone and in any batch.

Rounding: against 80-bit values REF_COMPAT's error over a table's points (2-norm
over that of the values, root mean square over tables of all sizes of terms) is
2.2e-16 with terms, coefficients and exponentials rounded once each, 3.0e-16
with base-2 ones, rounded twice; the test's line is a fifth above the first.
"""
import numpy as np
import pytest

import oracle
from ima2p_amd import _lib as L
from ima2p_amd import sim

pytestmark = pytest.mark.gpu

REF_TOL = 4.5e-10 + 2e-11


def numpy_terms(tab, ns, nm, x):
    t = tab.astype(np.float64)
    cc, fc, hc = t[:, :ns], t[:, ns:2 * ns], t[:, 2 * ns:3 * ns]
    mc, fm = t[:, 3 * ns:3 * ns + nm], t[:, 3 * ns + nm:3 * ns + 2 * nm]
    th, m = x[:ns], x[ns:]
    return (-t[:, 4 * ns + 3 * nm + 1] + cc @ (np.log(2.0) - np.log(th)) - hc.sum(1)
            - (2 * fc) @ (1 / th) + mc @ np.log(m) - fm @ m)


def exact(p):
    top = p.max()
    w = np.exp(p - top)
    return np.log(len(p)) - (top + np.log(w.sum())), w.sum() ** 2 / (w * w).sum()


def points(rng, n, ns, nm):
    return np.column_stack([rng.uniform(1, 12, (n, ns)), rng.uniform(0.05, 2.0, (n, nm))])


def close(got, want, tol):
    assert abs(got - want) <= tol * max(1.0, abs(want)), (got, want)


@pytest.mark.parametrize("G", [1, 4, 15, 17, 63, 65, 128, 255, 257, 300, 513, 40000])
def test_rows(engine, G):
    rng = np.random.default_rng(G)
    tab = sim.lmode_table(rng, G)
    tid = engine.lmode_table(tab, 3, 2, 2)
    x = points(rng, 70, 3, 2)
    ex, ess = engine.jointp(tid, x, mode=L.LMODE_EXACT)
    rc, ess_rc = engine.jointp(tid, x, mode=L.LMODE_REF_COMPAT)
    for i in range(0, 70, 3):
        want, want_ess = exact(numpy_terms(tab, 3, 2, x[i]))
        close(ex[i], want, 2e-11)
        close(ess[i], want_ess, 1e-9)
        want, want_ess = oracle.jointp(tab, 3, 2, 2, x[i], ess=True)
        close(rc[i], want, REF_TOL)
        close(ess_rc[i], want_ess, 4 * REF_TOL)
    engine.lmode_free(tid)


@pytest.mark.parametrize("nr", range(1, 17))
def test_parameters(engine, nr):
    rng = np.random.default_rng(100 + nr)
    ns, nm = (nr + 1) // 2, nr // 2
    tab = sim.lmode_table(rng, 700, npsize=ns, nmig=nm, nsplit=1)
    tid = engine.lmode_table(tab, ns, nm, 2)
    x = points(rng, 35, ns, nm)
    ex, ess = engine.jointp(tid, x, mode=L.LMODE_EXACT)
    rc, _ = engine.jointp(tid, x, mode=L.LMODE_REF_COMPAT)
    for i in range(0, 35, 2):
        want, want_ess = exact(numpy_terms(tab, ns, nm, x[i]))
        close(ex[i], want, 2e-11)
        close(ess[i], want_ess, 1e-9)
        close(rc[i], oracle.jointp(tab, ns, nm, 2, x[i]), REF_TOL)
    engine.lmode_free(tid)


@pytest.mark.parametrize("shape", [(3, 2, 2, 0, (0, 5)), (5, 8, 3, 2, (5, 13)), (6, 5, 2, 0, (0, 11))])
def test_same_bits_in_any_batch(engine, shape):
    ns, nm, npops, model, pr = shape
    rng = np.random.default_rng(9)
    tid = engine.lmode_table(sim.lmode_table(rng, 70000, ns, nm, nsplit=npops - 1), ns, nm, npops)
    x = points(rng, 3000, ns, nm)
    for mode in (L.LMODE_EXACT, L.LMODE_REF_COMPAT):
        full = engine.jointp(tid, x, mode=mode, modeltype=model, prange=pr)
        for lo, n in ((0, 1), (5, 1), (0, 15), (1, 16), (3, 17), (10, 64), (7, 65), (100, 129),
                      (1000, 1025)):
            part = engine.jointp(tid, x[lo:lo + n], mode=mode, modeltype=model, prange=pr)
            for a, b in zip(part, full):
                np.testing.assert_array_equal(a, b[lo:lo + n])
    engine.lmode_free(tid)


# -log probabilities by row, as (offset below the top, rows): which values
# the running maximum keeps decides the list cap
WINDOWS = {
    "all_in": [(4.0, 5), (0.0, 1), (6.0, 700)],
    "first_out": [(20.0, 1), (3.0, 600), (0.0, 1)],
    "kept_out": [(5.0, 2), (14.0, 1), (3.0, 600), (0.0, 1), (7.0, 50)],
    "never_kept": [(5.0, 300), (16.0, 400), (0.0, 1), (12.0, 300)],
    "kept_in_a_later_stage": [(6.0, 1300), (15.5, 1), (4.0, 900), (0.0, 1)],
    "after_the_top": [(1.0, 40), (0.0, 1), (10.5, 900)],
    "one": [(0.0, 1)],
}


@pytest.mark.parametrize("name", sorted(WINDOWS))
def test_window_and_list_cap(engine, name):
    rng = np.random.default_rng(4)
    off = np.concatenate([d + rng.uniform(0, 0.4, n) * (d > 0) for d, n in WINDOWS[name]])
    tab = np.zeros((len(off), 4 * 1 + 3 * 1 + 2 + 1), np.float32)
    tab[:, 8] = off - 30.0  # probg; the counts and sums are zero
    tid = engine.lmode_table(tab, 1, 1, 2)
    x = np.array([[3.0, 0.5]])
    out, ess = engine.jointp(tid, np.tile(x, (20, 1)), mode=L.LMODE_REF_COMPAT)
    want, want_ess = oracle.jointp(tab, 1, 1, 2, x[0], ess=True)
    for i in range(20):
        close(out[i], want, REF_TOL)
        close(ess[i], want_ess, 4 * REF_TOL)
    engine.lmode_free(tid)


def test_values_that_are_not_finite(engine):
    rng = np.random.default_rng(12)
    base = sim.lmode_table(rng, 600)
    x = points(rng, 18, 3, 2)
    far = x.copy()
    far[3, 0] = 1e-308  # 2 / x overflows: that point's terms are all -inf
    tid = engine.lmode_table(base, 3, 2, 2)
    good, _ = engine.jointp(tid, x, mode=L.LMODE_EXACT)
    out, _ = engine.jointp(tid, far, mode=L.LMODE_EXACT)
    assert out[3] == np.inf
    np.testing.assert_array_equal(np.delete(out, 3), np.delete(good, 3))
    engine.lmode_free(tid)
    for value, where, want in ((np.inf, 3, "drop"), (np.nan, 3, "nan")):
        tab = base.copy()
        tab[300, where] = value  # a coalescent sum: its row's term is -inf or NaN
        tid = engine.lmode_table(tab, 3, 2, 2)
        out, _ = engine.jointp(tid, x, mode=L.LMODE_EXACT)
        if want == "nan":
            assert np.isnan(out).all()
        else:
            p = [np.delete(numpy_terms(base, 3, 2, q), 300) for q in x]
            for i in range(len(x)):
                close(out[i], exact(p[i])[0] + np.log(600 / 599), 2e-11)
        engine.lmode_free(tid)


def test_rounding(engine):
    ratio = []
    for seed in range(30):
        rng = np.random.default_rng(seed)
        tab = sim.lmode_table(rng, 3000) * np.float32(2.0 ** rng.uniform(-1.5, 1.5))
        x = np.column_stack([rng.uniform(0.5, 15, (30, 3)), rng.uniform(0.05, 4.0, (30, 2))])
        tid = engine.lmode_table(np.ascontiguousarray(tab), 3, 2, 2)
        out, _ = engine.jointp(tid, x, mode=L.LMODE_REF_COMPAT)
        engine.lmode_free(tid)
        t, v = tab.astype(np.longdouble), x.astype(np.longdouble)
        err, size = [], []
        cc, fc, hc, mc, fm = t[:, :3], t[:, 3:6], t[:, 6:9], t[:, 9:11], t[:, 11:13]
        for i in range(len(x)):
            p = (-t[:, 19] + cc @ (np.log(np.longdouble(2)) - np.log(v[i, :3])) - hc.sum(1)
                 - (2 * fc) @ (1 / v[i, :3]) + mc @ np.log(v[i, 3:]) - fm @ v[i, 3:])
            p = p[p > p.max() - 10]  # no list cap: values outside the window are kept first
            want = np.log(np.longdouble(3000)) - (p.max() + np.log(np.exp(p - p.max()).sum()))
            err.append(float(out[i] - want))
            size.append(float(want))
        ratio.append(np.linalg.norm(err) / np.linalg.norm(size))
    assert np.sqrt(np.mean(np.square(ratio))) <= 1.2 * 2.2e-16


def test_large_terms(engine):
    """Base terms beyond 1e22 take the careful path, with padding behind them;
    a term of -1.5e308 is still one."""
    rng = np.random.default_rng(2)
    for G in (1, 70, 300, 600, 40000):
        tab = sim.lmode_table(rng, G)
        x = points(rng, 20, 3, 2)
        tab[:, 19] = 1e30
        tid = engine.lmode_table(tab, 3, 2, 2)
        out, _ = engine.jointp(tid, x, mode=L.LMODE_EXACT)
        np.testing.assert_allclose(out, np.float64(np.float32(1e30)), rtol=1e-15)
        engine.lmode_free(tid)
    tab = np.zeros((1, 10), np.float32)
    tab[0, 1] = 1e38  # fc
    tid = engine.lmode_table(tab, 1, 1, 2)
    fc = np.float64(tab[0, 1])
    out, _ = engine.jointp(tid, np.array([[fc / 0.75e308, 1.0]]), mode=L.LMODE_EXACT)
    np.testing.assert_allclose(out, 1.5e308, rtol=1e-15)
    engine.lmode_free(tid)


@pytest.mark.parametrize("row", [3, 300, 99999])
def test_infinite_term_in_any_stage(engine, row):
    """Two stages a chunk: a term of +inf gives no number wherever it stands."""
    tab = sim.lmode_table(np.random.default_rng(3), 100000)
    tab[row, 19] = -np.inf
    tid = engine.lmode_table(tab, 3, 2, 2)
    out, _ = engine.jointp(tid, points(np.random.default_rng(4), 70, 3, 2), mode=L.LMODE_EXACT)
    assert np.isnan(out).all()
    engine.lmode_free(tid)
