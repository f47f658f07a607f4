"""Workloads for timing the engine through its Python front end.

Every case is one thing that a program using the engine has it do:

  plain    one likelihoodHKY-shaped call: a genealogy in host arrays is
           uploaded, scored in FP64 and its log-likelihood returned
  score    one batched ima_score over every (chain, locus) genealogy
  state    a whole chain state evaluated, as after loading a checkpoint:
           every locus scored and every chain's genealogy prior integrated
  sweep    sweeps of the Metropolis-coupled chains, the full step (the
           genealogy move, split-time and mutation-rate updates, the swap),
           then the chains' state read back
  joint    L-mode jointp at a batch of points over a genealogy table
  curves   L-mode marginal curves of every parameter, the marginal peaks,
           and the 2NM density of every migration rate

Inputs come from the package's simulator and the seed alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ima2p_amd import _lib as L
from ima2p_amd import immodel, sim, workloads
from ima2p_amd.engine import Engine
from ima2p_amd.serve import AnalysisSpec

QMAX, MMAX, TMAX = 20.0, 5.0, 5.0
STEP = (L.MC3_GRAPH | L.MC3_TOPOLOGY | L.MC3_SCALE | L.MC3_RY1 | L.MC3_UPDATE_U | L.MC3_NW)


def listed():
    return [
        # the smallest call: IMa2p's host code scores one proposal at a time
        {"name": "plain_one", "kind": "plain", "pops": 3, "copies": 45, "sites": 1000},
        # every genealogy of the 64-chain, 50-locus three-population analysis
        {"name": "score_3pop_fp32", "kind": "score", "pops": 3, "hky": 50, "infinite": 0, "step": 0,
         "low": 15, "high": 15, "short": 1000, "long": 1000, "chains": 64, "fp64": False},
        # uneven loci of all three mutation models, likelihoods and prior in FP64
        {"name": "state_mixed_fp64", "kind": "state", "pops": 2, "hky": 30, "infinite": 20, "step": 10,
         "low": 2, "high": 30, "short": 200, "long": 3000, "chains": 32, "fp64": True},
        # the reference's small run: 4 chains, 5 infinite-sites loci of 10 + 10 copies
        {"name": "sweep_2pop_small_fp64", "kind": "sweep", "pops": 2, "hky": 0, "infinite": 5, "step": 0,
         "low": 10, "high": 10, "short": 0, "long": 0, "chains": 4, "fp64": True, "sweeps": 50},
        # the headline analysis: 64 heated chains, 50 loci x 1000 bp, 45 copies
        {"name": "sweep_3pop_fp32", "kind": "sweep", "pops": 3, "hky": 50, "infinite": 0, "step": 0,
         "low": 15, "high": 15, "short": 1000, "long": 1000, "chains": 64, "fp64": False, "sweeps": 10},
        # an analysis as the request loop takes them: 4 populations, mixed loci
        {"name": "sweep_4pop_mixed_fp32", "kind": "sweep", "pops": 4, "hky": 20, "infinite": 13, "step": 7,
         "low": 2, "high": 10, "short": 200, "long": 1500, "chains": 32, "fp64": False, "sweeps": 10},
        # the uneven batch: 256 chains x 300 loci of 4 to 60 copies
        {"name": "sweep_uneven_fp32", "kind": "sweep", "pops": 2, "hky": 150, "infinite": 100, "step": 50,
         "low": 2, "high": 30, "short": 200, "long": 3000, "chains": 256, "fp64": False, "sweeps": 5},
        # one point of a resident table: a line search's step, the smallest query
        {"name": "joint_one_point", "kind": "joint", "sizes": 3, "rates": 2, "rows": 100000,
         "points": 1, "model": 0, "ref": False},
        # a generation of the joint-peak search: 100 vectors per parameter
        {"name": "joint_500_ref", "kind": "joint", "sizes": 3, "rates": 2, "rows": 100000,
         "points": 500, "model": 0, "ref": True},
        # a served query on a three-population table: its eight migration rates
        {"name": "joint_3pop_rates", "kind": "joint", "sizes": 5, "rates": 8, "rows": 30000,
         "points": 60, "model": 2, "ref": False},
        # a slice of a surface over the largest resident table
        {"name": "joint_surface", "kind": "joint", "sizes": 3, "rates": 2, "rows": 1000000,
         "points": 4096, "model": 0, "ref": False},
        # the marginal section of an L-mode report
        {"name": "curves_2pop", "kind": "curves", "sizes": 3, "rates": 2, "rows": 20000, "grid": 500},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["plain", "score", "state", "sweep", "sweep", "sweep", "joint", "joint", "joint", "curves"])
    if kind == "plain":
        return {"kind": kind, "pops": rng.randint(2, 4), "copies": _log_int(rng, 6, 120),
                "sites": rng.randint(200, 3000)}
    if kind == "joint":
        three = rng.random() < 0.3
        rows, points = _log_int(rng, 10000, 1000000), _log_int(rng, 1, 4096)
        return {"kind": kind, "sizes": 5 if three else 3, "rates": 8 if three else 2,
                "rows": rows // 2 if three else rows, "points": points,
                "model": rng.randint(1, 2) if three else 0, "ref": rng.random() < 0.5}
    if kind == "curves":
        return {"kind": kind, "sizes": 3, "rates": 2, "rows": _log_int(rng, 5000, 20000),
                "grid": rng.randint(100, 500)}
    pops = rng.randint(2, 4)
    loci, chains = _log_int(rng, 5, 150), _log_int(rng, 4, 128)
    hky = rng.choice([loci, loci // 2, loci // 2, 0])
    infinite = (loci - hky) * 2 // 3
    c = {"kind": kind, "pops": pops, "hky": hky, "infinite": infinite, "step": loci - hky - infinite,
         "low": rng.randint(2, 6), "high": rng.randint(6, 60 // pops), "short": rng.randint(200, 500),
         "long": rng.randint(600, 3000), "chains": chains, "fp64": rng.random() < 0.4}
    if kind == "sweep":
        c["sweeps"] = rng.randint(5, 10)
    return c


# --------------------------------------------------------------- inputs --

def _analysis(case, seed):
    """Loci simulated under a random model of `pops` populations; the chains
    start on the genealogies that generated the data and, at loci without
    the infinite-sites restriction, on others of the same model."""
    rng = np.random.default_rng(seed)
    P = case["pops"]
    pt, theta, ts, mig = (sim.im_model_two_pop() if P == 2 else
                          sim.im_model_three_pop(rng) if P == 3 else sim.im_model_random(rng, P))
    model = immodel.build(pt, qmax=QMAX, mmax=MMAX)
    kinds = ["hky"] * case["hky"] + ["is"] * case["infinite"] + ["sw"] * case["step"]
    loci, samp, u, gens, states = [], [], [], [], []
    for kind in kinds:
        sp = [int(k) for k in rng.integers(case["low"], case["high"] + 1, P)]
        while True:
            g = sim.simulate_genealogy(rng, sp, theta, ts, mig, pt)
            pool, A = [g], None
            if kind == "hky":
                uu = float(rng.lognormal(0.0, 0.5))
                nsites = int(rng.integers(case["short"], case["long"] + 1))
                data = sim.encode_hky(sim.simulate_hky_sequences(
                    rng, g, nsites, rng.dirichlet([10] * 4), 4.0, uu))
                pool.append(sim.simulate_genealogy(rng, sp, theta, ts, mig, pt))
            elif kind == "is":
                uu = float(rng.uniform(0.5, 2.0))
                data = sim.simulate_is(rng, g, uu)
                if data.seq.shape[1] == 0:
                    continue
            else:
                uu = float(rng.uniform(0.5, 2.0))
                A = sim.simulate_sw(rng, g, uu, start=20)
                data = g.n
            break
        loci.append((kind, data))
        samp.append(sp)
        u.append(uu)
        gens.append(pool)
        states.append(A)
    C = case["chains"]
    kappa = np.array([4.0 if k == "hky" else 1.0 for k in kinds])
    return AnalysisSpec(
        loci=loci, model=model, samppop=samp, chains=[[p[c % len(p)] for p in gens] for c in range(C)],
        u=np.tile(u, (C, 1)), kappa=np.tile(kappa, (C, 1)), beta=workloads.geometric_betas(C),
        tvals=np.tile(np.asarray(ts, float), (C, 1)), tmax=TMAX, seed=seed % (1 << 30) + 1,
        precision=L.PREC_FP64 if case["fp64"] else L.PREC_FP32, A=[states] * C)


def _table(case, seed):
    """Genealogy summaries and points over the bulk of the priors."""
    rng = np.random.default_rng(seed)
    ns, nr = case["sizes"], case["rates"]
    table = sim.lmode_table(rng, case["rows"], ns, nr, nsplit=1 if ns == 3 else 2)
    if case["kind"] == "curves":
        return table, None
    x = np.concatenate([rng.uniform(1.0, 10.0, (case["points"], ns)),
                        rng.uniform(0.05, 2.0, (case["points"], nr))], axis=1)
    return table, x


def _range(case):
    ns, nr = case["sizes"], case["rates"]
    return [(0, ns + nr), (0, ns), (ns, ns + nr)][case["model"]]


def _plain(case, seed):
    rng = np.random.default_rng(seed)
    P = case["pops"]
    pt, theta, ts, mig = sim.im_model_two_pop() if P == 2 else sim.im_model_random(rng, P)
    n = case["copies"]
    sp = [n // P + (1 if i < n % P else 0) for i in range(P)]
    g = sim.simulate_genealogy(rng, sp, theta, ts, mig, pt)
    u = float(rng.lognormal(0.0, 0.5))
    data = sim.encode_hky(sim.simulate_hky_sequences(rng, g, case["sites"], rng.dirichlet([10] * 4), 4.0, u))
    return data, sim.simulate_genealogy(rng, sp, theta, ts, mig, pt), u


def prepare(case, seed):
    e = Engine(0)
    s = {"case": case, "engine": e}
    kind = case["kind"]
    if kind == "plain":
        data, s["tree"], s["u"] = _plain(case, seed)
        s["locus"] = e.add_locus_hky(data)
    elif kind in ("joint", "curves"):
        table, s["x"] = _table(case, seed)
        s["table"] = e.lmode_table(table, case["sizes"], case["rates"], 2 if case["sizes"] == 3 else 3)
        if kind == "curves":
            n = case["grid"]
            s["size_axis"] = QMAX * (np.arange(n) + 0.5) / n
            s["rate_axis"] = MMAX * (np.arange(n) + 0.5) / n
            s["flow_axis"] = 0.5 * QMAX * MMAX * (np.arange(n) + 0.5) / n
    else:
        spec = _analysis(case, seed)
        first, _ = spec.load(e)
        s["spec"], s["first"] = spec, first
        if kind != "sweep":
            n = spec.nchains * spec.nloci
            s["items"] = e.items(first + np.arange(n), spec.u.ravel(), spec.kappa.ravel())
            s["groups"] = [first + c * spec.nloci + np.arange(spec.nloci) for c in range(spec.nchains)]
    return s


def run(s):
    e, case = s["engine"], s["case"]
    kind = case["kind"]
    if kind == "plain":
        return e.likelihood_hky(s["locus"], s["tree"], s["u"], 4.0)
    if kind == "joint":
        return e.jointp(s["table"], s["x"], mode=L.LMODE_REF_COMPAT if case["ref"] else L.LMODE_EXACT,
                        modeltype=case["model"], prange=_range(case))
    if kind == "curves":
        ns, nr, t = case["sizes"], case["rates"], s["table"]
        curves, peaks, flow = [], [], []
        for p in range(ns + nr):
            curves.append(e.margincalc(t, p, s["size_axis"] if p < ns else s["rate_axis"]))
            peaks.append(e.marginal_peak(t, p, 1e-7, QMAX if p < ns else MMAX)[:2])
        for m in range(nr):
            flow.append(e.popmig(t, m, m, s["flow_axis"], QMAX, MMAX))
        return {"curves": np.stack(curves), "peaks": np.array(peaks), "flow": np.stack(flow)}
    spec = s["spec"]
    if kind in ("score", "state"):
        like, status = e.score(s["items"], spec.precision)
        if kind == "score":
            return {"like": like, "status": status}
        probg, q, m = e.prior(s["groups"], spec.tvals, spec.model)
        return {"like": like, "status": status, "probg": probg, "sizes": q, "rates": m}
    e.mc3_run(case["sweeps"], STEP)
    pdg, beta, _, _ = e.mc3_read()
    probg, tvals = e.mc3_read_prior()
    u, kappa = e.mc3_read_rates()
    return {"pdg": pdg, "beta": beta, "probg": probg, "splits": tvals, "u": u, "kappa": kappa}


# ------------------------------------------------------------ the work --

def work(case):
    """Likelihood flops: (36 n - 58) per site pattern, about one pattern for
    20 sites, plus the prior's and the moves' few operations per event; a
    sweep scores each genealogy 1.65 times (the proposal, a quarter of a
    time update, 0.4 of a mutation-rate round).  L mode: 2 fused
    multiply-adds per parameter and an exp of about 20 operations per
    (point, genealogy) pair; a 2NM density term is about 150."""
    kind = case["kind"]
    if kind == "plain":
        n, S = case["copies"], 10 + case["sites"] / 25
        return {"bytes": (2 * n - 1) * 20 + n * S, "flops": (36 * n - 58) * S}
    if kind in ("joint", "curves"):
        ns, nr, G = case["sizes"], case["rates"], case["rows"]
        K = 4 * ns + 3 * nr + 3
        if kind == "joint":
            r0, r1 = _range(case)
            # one base value, then a count and a sum per parameter in range
            return {"bytes": 4 * G * (1 + 2 * (r1 - r0)) + case["points"] * 8 * (ns + nr + 2),
                    "flops": case["points"] * G * (4.0 * (r1 - r0) + 24)}
        pts = (ns + nr) * (case["grid"] + 1024 + 100)
        return {"bytes": 4 * G * K, "flops": G * (26.0 * pts + 150.0 * nr * case["grid"])}
    loci = case["hky"] + case["infinite"] + case["step"]
    n = case["pops"] * (case["low"] + case["high"]) / 2
    S = 10 + (case["short"] + case["long"]) / 50
    items = case["chains"] * loci
    events = 2 * n
    like = case["chains"] * ((36 * n - 58) * S * case["hky"] + 30 * n * (loci - case["hky"]))
    genealogy = (2 * n - 1) * 24 + events / 2 * 16
    if kind == "sweep":
        k = case["sweeps"]
        return {"bytes": k * items * 2 * genealogy, "flops": k * (1.65 * like + items * 40 * events)}
    return {"bytes": items * (genealogy + 12) + loci * n * S,
            "flops": like + (items * 20 * events if kind == "state" else 0)}


def tolerance(case):
    """About four times what was seen between two correct evaluations: FP32
    pruning against FP64 for single-precision scores, FP64 sums in another
    order for the rest (with 1e-10 for the Bessel polynomials, and 1e-7 for
    the golden section of a flat-topped peak)."""
    kind = case["kind"]
    if kind in ("plain", "joint"):
        return {"rel": 1e-12}
    if kind == "curves":
        return {"rel": 1e-6, "max": 1e-5}
    if kind in ("score", "state"):
        return {"rel": 3e-10} if case["fp64"] else {"rel": 3e-7, "max": 2e-6}
    # a chain whose FP32 likelihood rounds another way may take another
    # decision (seldom: 1 in 1e6) and differs from then on: FP64-scored sweeps
    # of the uneven batch end up to 3e-3 from FP32-scored ones
    return {"rel": 1e-9} if case["fp64"] else {"rel": 0.012, "max": 0.9}


# ------------------------------------------------- the results in 64 bits --

def _lengths(g):
    t = np.asarray(g.time, float)
    up = np.asarray(g.up0)
    return np.where(up < 0, t, t - t[np.maximum(up, 0)])


def _order(g):
    """Internal nodes, daughters before parents."""
    inner = np.arange(g.n, 2 * g.n - 1)
    return inner[np.argsort(np.asarray(g.time)[np.asarray(g.up0)[inner]], kind="stable")]


def _hky(g, data, u, kappa):
    pi = np.asarray(data.pi, float)
    cls = np.array([pi[0] + pi[2], pi[1] + pi[3]] * 2)
    same = np.eye(4)
    ts = np.array([[float((i + j) % 2 == 0) for j in range(4)] for i in range(4)]) - same
    rate = u / (data.totsites * (pi @ (ts * kappa + (1 - same - ts)) @ pi))
    d = rate * _lengths(g)[:, None, None]
    e, ea = np.exp(-d), np.exp(-d * (1 + cls * (kappa - 1)))
    P = (pi * (1 - e) * (1 - same - ts)
         + (same + ts) * (pi + pi * e * (1 / cls - 1))
         + ea * (same * (cls - pi) / cls - ts * pi / cls))
    part, scale = {}, np.zeros(data.seq.shape[1])
    for v in _order(g):
        f = 1.0
        for d in (int(g.up0[v]), int(g.up1[v])):
            f = f * (P[d][:, data.seq[d]] if d < g.n else P[d] @ part.pop(d))
        m = f.max(axis=0)
        scale += np.log(m)
        part[v] = f / m
    return float(data.mult @ (np.log(pi @ part[g.root]) + scale))


def _bessel(k, x):
    """exp(-x) I_k(x) by its power series, summed in logarithms."""
    k = np.abs(k)[:, None].astype(float)
    m = np.arange(0, 400)[None, :]
    lg = torch.lgamma(torch.from_numpy(m + 1.0)) + torch.lgamma(torch.from_numpy(m + k + 1.0))
    t = (2 * m + k) * np.log(x[:, None] / 2) - lg.numpy() - x[:, None]
    top = t.max(axis=1)
    return top + np.log(np.exp(t - top[:, None]).sum(axis=1))


def _step(g, A, u):
    keep = np.asarray(g.down) >= 0
    d = np.asarray(A)[keep] - np.asarray(A)[np.asarray(g.down)[keep]]
    return float(_bessel(d, _lengths(g)[keep] * u).sum())


def _infinite(g, data, u):
    """Every site's mutation lies on the branch above its clade; the clade of
    a root's daughter is the complement of its sister's and both count.  The
    constant counts the mutations of each node's two daughter branches."""
    n, ln = g.n, _lengths(g)
    clade = [1 << i if i < n else 0 for i in range(2 * n - 1)]
    for v in _order(g):
        clade[v] = clade[int(g.up0[v])] | clade[int(g.up1[v])]
    where = {}
    full = (1 << n) - 1
    for v in range(2 * n - 1):
        if g.down[v] < 0:
            continue
        t = ln[v]
        if g.down[v] == g.root:
            t = ln[int(g.up0[g.root])] + ln[int(g.up1[g.root])]
        where[clade[v]] = where[full ^ clade[v]] = t, int(g.down[v])
    p = -u * float(ln[np.asarray(g.down) >= 0].sum())
    counts = {}
    for site in data.seq.T:
        key = sum(1 << i for i in np.flatnonzero(site).tolist())
        t, node = where[key]
        p += math.log(t * u)
        counts[node] = counts.get(node, 0) + 1
    return p - sum(math.lgamma(c + 1) for c in counts.values())


def _weights(g, model, ts, samp):
    """Coalescent and migration counts and time sums by (period, position)."""
    P, n = model.npops, g.n
    ev = [(float(g.time[g.up0[v]]), 0, v, 0) for v in range(n, 2 * n - 1)]
    for v in range(2 * n - 1):
        ev += [(float(t), 1, v, int(to)) for t, to in g.mig[v]]
    root = max(e[0] for e in ev if e[1] == 0)
    ev += [(float(t), 2, k, 0) for k, t in enumerate(ts) if t <= root]
    ev.sort(key=lambda e: e[0])
    pop = {v: int(g.pop[v]) for v in range(n)}  # the lineages and where they are
    num = np.zeros(2 * P - 1)
    num[:P] = samp
    cc, fc = np.zeros((P, P)), np.zeros((P, P))
    mc, fm = np.zeros((P, P, P)), np.zeros((P, P, P))
    k, last = 0, 0.0
    for t, what, v, to in ev:
        here = list(model.plist[k][:model.npresent[k]])
        dt, last = t - last, t
        for i, p in enumerate(here):
            fc[k, i] += num[p] * (num[p] - 1) * dt / 2
            if k < P - 1:
                fm[k, i, :len(here)] += num[p] * dt
        if what == 0:
            p = pop.pop(int(g.up0[v]))
            pop.pop(int(g.up1[v]))
            pop[v] = p
            cc[k, here.index(p)] += 1
            num[p] -= 1
        elif what == 1:
            mc[k, here.index(pop[v]), here.index(to)] += 1
            num[pop[v]] -= 1
            num[to] += 1
            pop[v] = to
        else:
            a, b, new = (int(q) for q in model.join[k])
            num[new], num[a], num[b] = num[a] + num[b], 0, 0
            pop = {v: new if p in (a, b) else p for v, p in pop.items()}
            k += 1
    return cc, fc, mc, fm


_NODES, _PESO = np.polynomial.legendre.leggauss(16)


def _integral(log_f, top):
    """log of the integral of exp(log_f(x)) over (0, top): Gauss-Legendre in
    log x, panels of 0.1 over the last 60 units."""
    edge = math.log(top) - np.arange(600, -1, -1) * 0.1
    s = (edge[:-1, None] + edge[1:, None] + 0.1 * _NODES[None, :]) / 2
    v = log_f(np.exp(s)) + s
    m = v.max()
    return float(m + math.log((np.exp(v - m) * (0.05 * _PESO)).sum()))


def _prior(spec, c, cache):
    total = None
    for l, g in enumerate(spec.chains[c]):
        key = (l, id(g))
        if key not in cache:
            cache[key] = _weights(g, spec.model, spec.tvals[c], spec.samppop[l])
        total = cache[key] if total is None else tuple(a + b for a, b in zip(total, cache[key]))
    cc, fc, mc, fm = total
    q, m = [], []
    for wp in spec.model.theta_wp:
        n, f = sum(cc[k, i] for k, i in wp), sum(fc[k, i] for k, i in wp)
        q.append(_integral(lambda x: n * np.log(2 / x) - 2 * f / x, QMAX))
    for wp in spec.model.mig_wp:
        n, f = sum(mc[k, i, j] for k, i, j in wp), sum(fm[k, i, j] for k, i, j in wp)
        m.append(_integral(lambda x: n * np.log(x) - f * x, MMAX))
    return q, m


def exact(case, seed):
    kind = case["kind"]
    if kind == "plain":
        data, g, u = _plain(case, seed)
        return _hky(g, data, u, 4.0)
    if kind in ("joint", "curves"):
        ns, nr, G = case["sizes"], case["rates"], case["rows"]
        points = case["points"] if kind == "joint" else 2 * case["grid"]
        if points * G > 5e8:
            return None
        table, x = _table(case, seed)
        t = torch.from_numpy(table).double()
        cut = np.cumsum([0, ns, ns, ns, nr, nr, ns, nr, 1, 1])
        cc, fc, hc, mc, fm, qi, mi, _, probg = (t[:, a:b] for a, b in zip(cut[:-1], cut[1:]))
        if kind == "joint":
            base = -probg[:, 0] if ns == 3 else -qi.sum(1) if case["model"] == 1 else -mi.sum(1)
            r0, r1 = _range(case)
            out, ess = [], []
            for block in torch.from_numpy(x).split(64):
                p = base[:, None].expand(-1, len(block)).clone()
                for i in range(r0, r1):
                    v = block[:, i]
                    if i < ns:
                        p += cc[:, i, None] * (math.log(2.0) - v.log()) - hc[:, i, None] - 2 * fc[:, i, None] / v
                    else:
                        p += mc[:, i - ns, None] * v.log() - fm[:, i - ns, None] * v
                if case["ref"]:  # values within 10 nats of the largest
                    p[p <= p.max(0).values - 10] = -math.inf
                lse = torch.logsumexp(p, 0)
                out.append(math.log(G) - lse)
                ess.append((2 * lse - torch.logsumexp(2 * p, 0)).exp())
            return torch.cat(out).numpy(), torch.cat(ess).numpy()
        n, curves = case["grid"], []
        at = torch.from_numpy((np.arange(n) + 0.5) / n)
        for i in range(ns + nr):
            if i < ns:
                v = at * QMAX
                p = -qi[:, i] - hc[:, i], cc[:, i], math.log(2.0) - v.log(), fc[:, i], -2 / v
            else:
                v = at * MMAX
                p = -mi[:, i - ns], mc[:, i - ns], v.log(), fm[:, i - ns], -v
            f = p[0][:, None] + p[1][:, None] * p[2] + p[3][:, None] * p[4]
            curves.append(torch.logsumexp(f, 0) - math.log(G))
        return {"curves": torch.stack(curves).numpy(), "peaks": None, "flow": None}
    if kind == "sweep":
        return None
    spec = _analysis(case, seed)
    if spec.nchains * case["hky"] > 10000 or spec.nloci * case["high"] > 10000:
        return None
    cache, like = {}, np.zeros((spec.nchains, spec.nloci))
    for c in range(spec.nchains):
        for l, (what, data) in enumerate(spec.loci):
            g = spec.chains[c][l]
            key = (l, id(g))
            if key not in cache:
                u = spec.u[c, l]
                cache[key] = (_hky(g, data, u, 4.0) if what == "hky" else
                              _infinite(g, data, u) if what == "is" else _step(g, spec.A[c][l], u))
            like[c, l] = cache[key]
    if kind == "score":
        return {"like": like.ravel(), "status": None}
    seen = {}
    both = [_prior(spec, c, seen) if c < 2 or spec.model.npops > 1 else None for c in range(spec.nchains)]
    q, m = np.array([b[0] for b in both]), np.array([b[1] for b in both])
    return {"like": like.ravel(), "status": None, "probg": q.sum(1) + m.sum(1), "sizes": q, "rates": m}
