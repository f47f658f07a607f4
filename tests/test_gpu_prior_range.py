"""The integrals of the genealogy prior over the range of their arguments,
and the accept step's decisions for models of every size.

Integrals: counts from none to thousands, weights from far below to far
above the priors' bounds (either end of the incomplete gammas: series,
continued fraction, saturated), against the oracle.  Bound: both stop their
series at the same term (relative 3e-7, the comparison rounds at 1e-16), and
the logarithms of at most 1e5 in size that make an integral are within an ulp,
so the values agree to 1e-15 of the largest of them; the tolerance is the
path's own 1e-10 relative, with 1e-9 absolute for values near zero.

Logarithm: a migration rate without events and with weight f far above 1 /
its bound integrates to -log f exactly as the device takes the logarithm,
which must lie within an ulp of it.

Two coalescences of weight f over [0, max], 2 f / max >= 2: the fraction ends
at its first term, and the integral is log 2 - log f - 2 f / max, through the
logarithms of f and of the gamma's argument.  Rounding as written with an
exact logarithm gives 0.443 ulp root mean square at max = 20, the argument's
logarithm pieced together from others 0.515.

Decisions: for 2 to 5 populations (up to 326 weight entries, 44 parameters)
group sizes give the same sweeps bit for bit, and probg is the oracle's.
"""
import numpy as np
import pytest

import oracle
from ima2p_amd import _lib as L
from ima2p_amd import immodel, sim
from ima2p_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qmax,mmax", [(20.0, 5.0), (0.5, 0.01), (1000.0, 200.0)])
def test_integrals(engine, qmax, mmax):
    pt, theta, ts, mig = sim.im_model_two_pop()
    model = immodel.build(pt, qmax=qmax, mmax=mmax)
    mid = engine.model_add(model)
    P, R = 2, 3 * 4 + 2 * 8 + 1
    counts = [0, 1, 2, 3, 7, 40, 300, 2500]
    weights = np.concatenate([10.0 ** np.arange(-9.0, 7.0, 1.0),
                              [0.37, 3.1, 19.9, 20.0, 41.0, 299.0, 2499.0, 2502.0]])
    rec, want = [], []
    for c in counts:
        for f in weights:
            r = np.zeros(R)
            cc, fc = r[:4].reshape(2, 2), r[4:8].reshape(2, 2)
            mc, fm = r[12:20].reshape(2, 2, 2), r[20:28].reshape(2, 2, 2)
            k, i = model.theta_wp[0][0]
            cc[k, i], fc[k, i] = c, f
            k, i = model.theta_wp[1][0]
            cc[k, i], fc[k, i] = 3, 4.0
            k, i, j = model.mig_wp[0][0]
            mc[k, i, j], fm[k, i, j] = c, f
            rec.append(r)
            w = {"cc": cc.astype(int), "fc": fc, "hcc": np.zeros((2, 2)), "mc": mc.astype(int),
                 "fm": fm}
            want.append(oracle.integrate_tree_prob([w], model))
    rec = np.ascontiguousarray(rec)
    n = len(rec)
    q, m, pg = np.zeros((n, model.npsize)), np.zeros((n, model.nmig)), np.zeros(n)
    dp = lambda a: a.ctypes.data_as(L.dp)  # noqa: E731
    engine._chk(engine.lib.ima_integrate_tree_prob(engine.h, mid, dp(rec), n, dp(pg), dp(q), dp(m)),
                "integrate_tree_prob")
    for x in range(n):
        np.testing.assert_allclose(q[x], want[x][1], rtol=1e-10, atol=1e-9, err_msg=str(rec[x]))
        np.testing.assert_allclose(m[x], want[x][2], rtol=1e-10, atol=1e-9, err_msg=str(rec[x]))


def test_logarithm_within_an_ulp(engine):
    pt, theta, ts, mig = sim.im_model_two_pop()
    model = immodel.build(pt, qmax=20.0, mmax=1e8)  # f mmax > 710: e^(-f mmax) drops out
    mid = engine.model_add(model)
    rng = np.random.default_rng(5)
    f = np.concatenate([rng.uniform(0.5, 2.0, 60000), np.exp(rng.uniform(-11.0, 40.0, 20000)),
                        1.0 + np.ldexp(rng.uniform(-1.0, 1.0, 20000), -rng.integers(1, 50, 20000))])
    rec = np.zeros((len(f), 3 * 4 + 2 * 8 + 1))
    k, i, j = model.mig_wp[0][0]
    rec[:, 20 + (k * 2 + i) * 2 + j] = f
    n = len(rec)
    q, m, pg = np.zeros((n, model.npsize)), np.zeros((n, model.nmig)), np.zeros(n)
    dp = lambda a: a.ctypes.data_as(L.dp)  # noqa: E731
    for lo in range(0, n, 1000):
        r = np.ascontiguousarray(rec[lo:lo + 1000])
        engine._chk(engine.lib.ima_integrate_tree_prob(
            engine.h, mid, dp(r), len(r), dp(pg[lo:]), dp(q[lo:]), dp(m[lo:])),
            "integrate_tree_prob")
    want = -np.log(f.astype(np.longdouble))
    assert np.all(np.abs(m[:, 0] - want) <= np.spacing(np.abs(want).astype(np.float64)))


def test_two_coalescences_round_as_written(engine):
    pt, theta, ts, mig = sim.im_model_two_pop()
    model = immodel.build(pt, qmax=20.0, mmax=5.0)
    mid = engine.model_add(model)
    f = np.random.default_rng(6).uniform(20.0, 60.0, 40000)
    rec = np.zeros((len(f), 3 * 4 + 2 * 8 + 1))
    k, i = model.theta_wp[0][0]
    rec[:, k * 2 + i] = 2
    rec[:, 4 + k * 2 + i] = f
    n = len(rec)
    q, m, pg = np.zeros((n, model.npsize)), np.zeros((n, model.nmig)), np.zeros(n)
    dp = lambda a: a.ctypes.data_as(L.dp)  # noqa: E731
    engine._chk(engine.lib.ima_integrate_tree_prob(engine.h, mid, dp(rec), n, dp(pg), dp(q), dp(m)),
                "integrate_tree_prob")
    F = f.astype(np.longdouble)
    want = np.log(np.longdouble(2)) - np.log(F) - 2 * F / 20
    off = ((q[:, 0] - want) / np.spacing(np.abs(want).astype(np.float64))).astype(np.float64)
    assert np.sqrt((off ** 2).mean()) <= 1.05 * 0.443


def _chains(P, C_, Lc, seed):
    rng = np.random.default_rng(seed)
    pt, theta, ts, mig = sim.im_model_two_pop() if P == 2 else sim.im_model_random(rng, P)
    model = immodel.build(pt, qmax=20.0, mmax=5.0)
    samp = [3] * P
    e = Engine(0)
    mid = e.model_add(model)
    lids, base = [], []
    for _ in range(Lc):
        g = sim.simulate_genealogy(rng, samp, theta, ts, mig, pt)
        loc = sim.encode_hky(sim.simulate_hky_sequences(rng, g, 200, [0.25] * 4, 4.0, 2.0))
        lid = e.add_locus_hky(loc)
        e.locus_set_model(lid, mid, samp)
        lids.append(lid)
        base.append(g)
    first = e.alloc_slots(lids * C_)
    e.write_slots(first, base * C_)
    e.write_pops(first, base * C_)
    e.mc3_setup(C_, Lc, first, 2.0, 4.0, np.array([0.97 ** c for c in range(C_)]), seed=seed,
                precision=L.PREC_FP64)
    e.mc3_set_prior(np.tile(ts, (C_, 1)), 10.0, P)
    return e, model, first, Lc


@pytest.mark.parametrize("P", [2, 3, 4, 5])
def test_decisions(P):
    out = []
    for D in (1, 2, 4, 6):
        e, model, first, Lc = _chains(P, 3, 13, 70 + P)
        if D > e.mc3_prior_group():
            e.close()
            continue
        e.mc3_prior_group(D)
        e.mc3_run(16, L.MC3_GRAPH | L.MC3_SCALE | L.MC3_RY1 | L.MC3_TOPOLOGY | L.MC3_NW)
        pdg, beta, stats, _ = e.mc3_read()
        probg, tv = e.mc3_read_prior()
        slots = [first + c * Lc + np.arange(Lc) for c in range(3)]
        fresh, _, _ = e.prior(slots, tv, model)
        np.testing.assert_allclose(probg, fresh, rtol=1e-9)
        assert 0 < stats[1] < stats[0]
        out.append((pdg, beta, probg, tv, stats))
        e.close()
    assert len(out) > 1
    for other in out[1:]:
        for a, b in zip(out[0], other):
            np.testing.assert_array_equal(a, b)
