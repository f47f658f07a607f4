"""L-mode marginal curves and the searches on them, where the device splits
the work: tables of one row, a workgroup's rows and one more or less, several
rows a lane; one point, a tile of points and one more or less, the batch sizes
where a workgroup takes more points or the lanes change from rows to points.

* margincalc against its formula in NumPy FP64: a term's argument, a sum of
  parts up to a few hundred, is within 4 roundings of each (1e-13), and the
  sum's order gives less: 1e-12.  A point's value must have the same bits in
  every batch.
* popmig: both layouts add the same tree of terms, so a point's value must have
  the same bits in every batch.  The test of batches of 100 against larger
  ones allows for the same positive terms in another order (G * 2^-52, twice
  that for the exponential prior's changes of reference) with another rounding
  of a term's log: parts up to 500, ten of them, 10 * 500 * 2^-53 = 6e-13.
* peaks and limits must equal, bit for bit, the searches run here one point
  at a time; 2NM peaks with the same number of points."""
import numpy as np
import pytest

from ima2p_amd import _lib as L
from ima2p_amd import sim

pytestmark = pytest.mark.gpu

NP, NM = 3, 2


def _table(rng, G):
    base = sim.lmode_table(rng, min(G, 4000), npsize=NP, nmig=NM)
    tab = np.tile(base, (-(-G // len(base)), 1))[:G].astype(np.float32)
    tab[:, 3 * NP + 2 * NM:4 * NP + 3 * NM] *= 0.05  # densities of order 1
    return np.ascontiguousarray(tab)


def _margin(tab, p, x, expo, mean):
    t = tab.astype(np.float64)
    i = p if p < NP else p - NP
    if p < NP:
        cc, fc, hc, qi = t[:, i], t[:, NP + i], t[:, 2 * NP + i], t[:, 3 * NP + 2 * NM + i]
        return np.array([np.exp(-qi + np.rint(cc) * np.log(2 / v) - hc - 2 * fc / v).mean()
                         for v in x])
    mc, fm, mi = t[:, 3 * NP + i], t[:, 3 * NP + NM + i], t[:, 4 * NP + 2 * NM + i]
    pri = (lambda v: -np.log(mean) - v / mean) if expo else (lambda v: 0.0)
    return np.array([np.exp(-mi + pri(v) + np.rint(mc) * np.log(v) - fm * v).mean() for v in x])


@pytest.mark.parametrize("G,nx", [(1, 3), (255, 1), (256, 16), (257, 17), (700, 500), (5000, 2),
                                  (66000, 125), (66000, 131), (20000, 414), (20000, 415),
                                  (66000, 260), (140000, 130)])
def test_margincalc(engine, G, nx):
    rng = np.random.default_rng(G + nx)
    tab = _table(rng, G)
    t = engine.lmode_table(tab, NP, NM, 3)
    x = rng.uniform(0.2, 4.0, nx)
    few = rng.choice(nx, min(nx, 6), replace=False)
    for p, expo in ((0, False), (2, False), (3, False), (4, True)):
        got = engine.margincalc(t, p, x, logi=0, expo=expo, mean=0.7)
        ref = _margin(tab, p, x[few], expo, 0.7)
        assert np.all(np.abs(got[few] - ref) <= 1e-12 * ref)
        for k in few:
            assert engine.margincalc(t, p, x[k], logi=0, expo=expo, mean=0.7)[0] == got[k]
    engine.lmode_table_free(t)


@pytest.mark.parametrize("G", [1, 15, 17, 256, 700, 20011])
@pytest.mark.parametrize("expo", [False, True])
def test_popmig_layouts_agree(engine, G, expo):
    rng = np.random.default_rng(G)
    t = engine.lmode_table(_table(rng, G), NP, NM, 3)
    qmax, mpr = 15.0, (0.8 if expo else 3.0)
    for nx in (256, 257, 400):
        x = np.sort(rng.uniform(0.05, 10.0, nx))
        for kw in ({}, {"kind": L.POPMIG_MARGIN, "first": 0, "last": G},
                   {"kind": L.POPMIG_MARGIN, "first": G // 3, "last": G}):
            a = engine.popmig(t, 0, 1, x, qmax, mpr, expo=expo, **kw)
            b = np.concatenate([engine.popmig(t, 0, 1, x[i:i + 100], qmax, mpr, expo=expo, **kw)
                                for i in range(0, nx, 100)])
            assert np.all(np.abs(a - b) <= (6e-13 + 2 * G * 2.0 ** -52) * np.abs(b))
    engine.lmode_table_free(t)


# one row, a chunk's edges, a few chunks, two rows a leaf; the layouts change at
# 128 points and with the wavefronts these make
@pytest.mark.parametrize("G", [1, 63, 65, 700, 5000, 70001])
@pytest.mark.parametrize("expo", [False, True])
def test_popmig_same_bits_in_any_batch(engine, G, expo):
    rng = np.random.default_rng(G)
    t = engine.lmode_table(_table(rng, G), NP, NM, 3)
    qmax, mpr = 15.0, (0.8 if expo else 3.0)
    x = rng.uniform(0.05, 10.0, 9000 if G <= 65 else 1500)
    for kw in ({"prob_or_like": 1}, {"kind": L.POPMIG_MARGIN, "first": G // 3, "last": G}):
        full = engine.popmig(t, 0, 1, x, qmax, mpr, expo=expo, **kw)
        for lo, n in ((0, 1), (7, 1), (0, 63), (1, 64), (3, 65), (5, 127), (5, 128), (9, 129),
                      (200, 255), (100, 256), (50, 700)):
            part = engine.popmig(t, 0, 1, x[lo:lo + n], qmax, mpr, expo=expo, **kw)
            np.testing.assert_array_equal(part, full[lo:lo + n])
    engine.lmode_table_free(t)


def test_popmig_more_points_than_a_launch_takes(engine):
    t = engine.lmode_table(_table(np.random.default_rng(8), 65536), NP, NM, 3)
    x = np.random.default_rng(9).uniform(0.05, 10.0, 2 * 4096 + 131)  # 4096 a launch
    full = engine.popmig(t, 0, 1, x, 15.0, 0.8, expo=True)
    for lo in (0, 4000, 4096, 8192, len(x) - 131):
        np.testing.assert_array_equal(engine.popmig(t, 0, 1, x[lo:lo + 131], 15.0, 0.8, expo=True),
                                      full[lo:lo + 131])
    engine.lmode_table_free(t)


def _peak_one_by_one(e, t, p, lower, upper):
    def f(v):
        return e.margincalc(t, p, v)[0]
    x = lower + (upper - lower) * np.arange(1024.0) / 1023
    y = e.margincalc(t, p, x)
    b = int(np.argmax(y))
    a, c = x[max(b - 1, 0)], x[min(b + 1, 1023)]
    gr = 0.61803398874989484820
    x1, x2 = c - gr * (c - a), a + gr * (c - a)
    f1, f2 = f(x1), f(x2)
    while abs(c - a) > 1e-7 * (abs(x1) + abs(x2)):
        if f1 > f2:
            c, x2, f2 = x2, x1, f1
            x1 = c - gr * (c - a)
            f1 = f(x1)
        else:
            a, x1, f1 = x1, x2, f2
            x2 = a + gr * (c - a)
            f2 = f(x2)
    peak, fp = (x1, f1) if f1 > f2 else (x2, f2)
    if y[b] > fp:
        peak, fp = x[b], y[b]
    out = [peak, fp]
    for lo, hi in ((lower, peak), (peak, upper)):
        fl, fh = f(lo), f(hi)
        if (fl - (fp - 1.92)) * (fh - (fp - 1.92)) > 0:
            out.append(-1.0)
            continue
        it = 0
        while it < 100 and hi - lo > 1e-9 * (hi + lo):
            mid = 0.5 * (lo + hi)
            fm = f(mid)
            if (fm - (fp - 1.92)) * (fl - (fp - 1.92)) <= 0:
                hi = mid
            else:
                lo, fl = mid, fm
            it += 1
        out.append(0.5 * (lo + hi))
    out.append(2.0 * (fp - f(1e-7)) if p >= NP else 0.0)
    return out


# tables on which the searches look six, two and one steps ahead
@pytest.mark.parametrize("G", [700, 1500000, 3000000])
def test_marginal_peaks_are_those_of_single_points(engine, G):
    t = engine.lmode_table(_table(np.random.default_rng(3), G), NP, NM, 3)
    for p, lo, hi in ((0, 1e-7, 20.0), (1, 1e-7, 0.01), (3, 1e-7, 5.0), (4, 0.5, 0.6)):
        assert list(engine.marginal_peak(t, p, lo, hi)) == _peak_one_by_one(engine, t, p, lo, hi)
    engine.lmode_table_free(t)


@pytest.mark.parametrize("G,expo", [(700, False), (700, True), (200000, False)])
def test_popmig_peak_is_that_of_single_points(engine, G, expo):
    e = engine
    t = e.lmode_table(_table(np.random.default_rng(4), G), NP, NM, 3)
    qmax, mpr = 15.0, (0.8 if expo else 3.0)
    upper = 20.0 * mpr if expo else qmax * mpr / 2.0
    def f(v):
        return e.popmig(t, 0, 1, v, qmax, mpr, expo=expo, kind=L.POPMIG_MARGIN, first=0, last=G)[0]
    w = upper / 100.0
    fb = e.popmig(t, 0, 1, 1e-7 + np.arange(100.0) * w, qmax, mpr, expo=expo,
                  kind=L.POPMIG_MARGIN, first=0, last=G)
    j = int(np.argmin(fb))
    if j == 0:
        ax, cx = 1e-7, 1e-7 + w
        bx = (ax + cx) / 2.0
    elif j == 99:
        ax, bx, cx = 1e-7 + 99.0 * w, 1e-7 + 98.0 * w, upper
    else:
        bx, cx, ax = 1e-7 + (j - 1.0) * w, 1e-7 + (j + 1.0) * w, 1e-7 + j * w
    r, n = 0.61803399, 102
    cg = 1.0 - r
    x0, x3 = ax, cx
    x1, x2 = (bx, bx + cg * (cx - bx)) if abs(cx - bx) > abs(bx - ax) else (bx - cg * (bx - ax), bx)
    f1, f2 = f(x1), f(x2)
    while abs(x3 - x0) > 1e-7 * (abs(x1) + abs(x2)) and n < 2100:
        if f2 < f1:
            x0, x1, f1 = x1, x2, f2
            x2 = r * x1 + cg * x3
            f2 = f(x2)
        else:
            x3, x2, f2 = x2, x1, f1
            x1 = r * x2 + cg * x0
            f1 = f(x1)
        n += 1
    want = (x1 if f1 < f2 else x2, -min(f1, f2), n)
    assert e.popmig_peak(t, 0, 1, qmax, mpr, expo=expo, last=G) == want
    e.lmode_table_free(t)
