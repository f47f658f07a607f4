"""Genealogy weights where the device's event lists end: two to 66 gene copies
with few and many migrations, so that the events fill no, one or several
chunks of 64 and any remainder of four, in one to four populations.  Bit for
bit against the oracle (same order, same arithmetic)."""
import numpy as np
import pytest

import oracle
from ima2p_amd import immodel, sim
from tests.test_gpu_prior import _load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,low,high", [(2, 1, 3), (2, 31, 33), (3, 1, 2), (3, 18, 22),
                                        (4, 2, 16)])
def test_event_counts(engine, P, low, high):
    rng = np.random.default_rng(10 * P + low)
    sizes = set()
    for rate in (0.05, 3.0):
        pt, theta, ts, mig = (sim.im_model_two_pop(t=0.9, m12=rate, m21=0.7 * rate) if P == 2 else
                              sim.im_model_three_pop(rng) if P == 3 else
                              sim.im_model_random(rng, P))
        model = immodel.build(pt)
        ts = np.asarray(ts, float)
        for _ in range(6):
            samp = [int(k) for k in rng.integers(low, high + 1, P)]
            gens = [sim.relabel_internal(sim.simulate_genealogy(rng, samp, theta, ts, mig, pt),
                                         rng) for _ in range(3)]
            first = _load(engine, model, gens, samp)
            got = engine.treeweight(np.arange(first, first + 3), ts, P)
            for i, g in enumerate(gens):
                ref = oracle.treeweight(g, model, ts, samp, 1.0)
                for k in ("cc", "mc", "fc", "fm", "hcc"):
                    np.testing.assert_array_equal(got[k][i], ref[k])
                assert got["length"][i] == ref["length"]
                root = g.time[g.up0[g.root]]
                sizes.add(g.n - 1 + sum(len(m) for m in g.mig) + int((ts < root).sum()))
    assert {s % 4 for s in sizes} == {0, 1, 2, 3}
    assert max(sizes) > 64 or high < 16
