"""Populations and migration events of genealogies, which only the device
holds: writes whose event regions follow each other, lie elsewhere, are empty
or single; edges nothing has written; and chains whose genealogies, moved by
the device's sweeps, later writes to other slots must leave as they are.
Everything is compared exactly."""
import numpy as np
import pytest

from ima2p_amd import _lib as L
from ima2p_amd import immodel, sim
from ima2p_amd.engine import Engine
from ima2p_amd.immodel import mig_arrays

pytestmark = pytest.mark.gpu


def _gene(rng, nmig, n=5):
    """A two-population genealogy carrying nmig events (order and labels are
    all the store looks at)."""
    pt, theta, ts, mig = sim.im_model_two_pop(t=0.9, m12=0.8, m21=0.6)
    g = sim.relabel_internal(sim.simulate_genealogy(rng, [3, n - 3], theta, ts, mig, pt), rng)
    ne = 2 * n - 1
    edges = rng.integers(0, ne, nmig)
    g.mig = [sorted((float(rng.uniform(0, 1)), int(rng.integers(0, 2)))
                    for _ in range(int((edges == e).sum()))) for e in range(ne)]
    return g


def _same(e, slot, g):
    me, mt, mo = mig_arrays(g)
    de, dt, do = e.read_mig_events(slot)
    assert np.array_equal(de, me) and np.array_equal(dt, mt) and np.array_equal(do, mo)
    assert np.array_equal(e.read_pops(slot, 1), g.pop)


# counts of the first write, of the second (slots whose events do not fit get
# a new region, so the second write's regions no longer follow each other)
@pytest.mark.parametrize("first,second", [
    ([3, 4, 5], [3, 4, 5]),              # in place, one block
    ([3, 4, 5], [3, 70, 5]),             # the middle one moves
    ([0, 0, 0], [2, 0, 65]),             # none before
    ([1, 2, 3], [0, 0, 0]),              # all taken away
    ([200, 1, 64], [1, 300, 64]),        # more than a wavefront's lanes
    ([7], [9]), ([7], [64]),             # one slot
])
def test_event_regions(first, second):
    rng = np.random.default_rng(5)
    e = Engine(0)
    mid = e.model_add(immodel.build(sim.PopTree.two_pop(), qmax=4.0, mmax=1.0))
    lid = e.add_locus_sw(5)
    e.locus_set_model(lid, mid, [3, 2])
    s0 = e.alloc_slots([lid] * (len(first) + 2))
    around = [_gene(rng, 6), _gene(rng, 6)]
    assert not e.read_pops(s0, len(first) + 2).any()
    e.write_pops(s0, [around[0]])
    e.write_pops(s0 + 1 + len(first), [around[1]])
    for counts in (first, second):
        gens = [_gene(rng, k) for k in counts]
        e.write_pops(s0 + 1, gens)
        for i, g in enumerate(gens):
            _same(e, s0 + 1 + i, g)
        _same(e, s0, around[0])
        _same(e, s0 + 1 + len(first), around[1])
    e.close()


def test_refused_write_changes_nothing():
    rng = np.random.default_rng(6)
    e = Engine(0)
    mid = e.model_add(immodel.build(sim.PopTree.two_pop(), qmax=4.0, mmax=1.0))
    lid = e.add_locus_sw(5)
    e.locus_set_model(lid, mid, [3, 2])
    s0 = e.alloc_slots([lid] * 2)
    gens = [_gene(rng, 4), _gene(rng, 4)]
    A = [np.arange(2 * g.n - 1, dtype=np.int32) for g in gens]
    e.write_slots(s0, gens, A=A)
    e.write_pops(s0, gens)
    before = e.read_slots(s0, 2)
    other = [_gene(rng, 90), _gene(rng, 4)]
    other[1].mig[2] = [(0.5, 7)]  # no such population
    with pytest.raises(Exception):
        e.write_pops(s0, other)
    other[1].root = 0  # a tip
    with pytest.raises(Exception):
        e.write_slots(s0, other, A=A)
    for i in range(2):
        _same(e, s0 + i, gens[i])
    for a, b in zip(before, e.read_slots(s0, 2)):
        assert np.array_equal(a, b)
    e.close()


@pytest.mark.parametrize("flags", [L.MC3_SCALE, L.MC3_SCALE | L.MC3_NW,
                                   L.MC3_SCALE | L.MC3_TOPOLOGY,
                                   L.MC3_SCALE | L.MC3_NW | L.MC3_TOPOLOGY | L.MC3_GRAPH])
def test_writes_beside_swept_chains(flags):
    """Chains swept, another slot written and read, more slots allocated, the
    chains swept again: the chains' genealogies and the run that follows are
    those of an engine without the writes."""
    rng = np.random.default_rng(7)
    pt, theta, ts, mig = sim.im_model_two_pop(t=0.9, m12=0.8, m21=0.6)
    model = immodel.build(pt, qmax=4.0, mmax=1.5)
    samp, C = [4, 3], 3
    gens = [sim.relabel_internal(sim.simulate_genealogy(rng, samp, theta, ts, mig, pt), rng)
            for _ in range(C)]
    extra = [sim.relabel_internal(sim.simulate_genealogy(rng, samp, theta, ts, mig, pt), rng)
             for _ in range(2)]
    loc = sim.HKYLocus(7, rng.integers(0, 4, (7, 3)).astype(np.int8), np.ones(3, np.int32), 3,
                       np.array([0.25] * 4))

    def state(e, first):
        out = list(e.read_slots(first, C)) + [e.read_pops(first, C)]
        for i in range(C):
            out += list(e.read_mig_events(first + i))
        return out + list(e.mc3_read_prior())

    def run(write):
        e = Engine(0)
        mid = e.model_add(model)
        lid = e.add_locus_hky(loc)
        e.locus_set_model(lid, mid, samp)
        first = e.alloc_slots([lid] * C)
        spare = e.alloc_slots([lid])
        e.write_slots(first, gens)
        e.write_pops(first, gens)
        e.mc3_setup(C, 1, first, np.ones(1), np.full(1, 2.0), np.linspace(1, 0.5, C), seed=11)
        e.mc3_set_prior(np.tile(ts, (C, 1)), 5.0, model.npops)
        e.mc3_run(12, flags)
        a = state(e, first)
        if write:
            e.write_slots(spare, extra[:1])
            e.write_pops(spare, extra[:1])
            more = e.alloc_slots([lid] * 40)
            e.write_slots(more + 39, extra[1:])
            e.write_pops(more + 39, extra[1:])
            for x, y in zip(a, state(e, first)):
                assert np.array_equal(x, y)
            _same(e, spare, extra[0])
            _same(e, more + 39, extra[1])
        e.mc3_run(12, flags)
        b = state(e, first)
        e.close()
        return a + b

    for x, y in zip(run(False), run(True)):
        assert np.array_equal(x, y)
