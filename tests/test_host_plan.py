"""Host-only planning of the sweep's per-chain prior kernels (no device).

ima_mc3_prior_plan returns the accept group size ima_mc3_set_prior picks
for a population model and the dynamic LDS of the per-chain kernels at that
size.  Every launch stays within 64 KiB of dynamic LDS, whatever the device
allows per workgroup: models of four and five populations, whose weight
records are 177 and 326 doubles long, get smaller groups instead of larger
launches.  The sizes are the reference's default parameter maps
(setup_iparams, initialize.cpp:202-760) for ladder trees of 2..5
populations.

ima_lmode_popmig_plan returns the 2NM density's split of a call's rows and
its work area: every row lies in a chunk and every partial in the area, for
the rows of the call and not of the table (a shorter range may make more
chunks: 16384 rows more than 16385).
"""
import ctypes as C

import pytest

from ima2p_amd import _lib as L
from ima2p_amd import immodel
from ima2p_amd.sim import PopTree


def _ladder(P):
    joins, cur = [], 0
    for k in range(P - 1):
        joins.append((cur, k + 1))
        cur = P + k
    return PopTree(P, joins)


def _plan(model):
    lib = L.load()
    loci, lds = C.c_int(), C.c_int64()
    rc = lib.ima_mc3_prior_plan(model.npops, model.npsize, sum(len(w) for w in model.theta_wp),
                                model.nmig, sum(len(w) for w in model.mig_wp),
                                C.byref(loci), C.byref(lds))
    return rc, loci.value, lds.value


@pytest.mark.parametrize("P", [1, 2, 3, 4, 5])
def test_group_size_fits_64k(P):
    model = immodel.build(_ladder(P) if P > 1 else PopTree(1, []))
    rc, loci, lds = _plan(model)
    assert rc == L.IMA_OK
    assert 1 <= loci <= 6
    assert 0 < lds <= 65536
    if P <= 3:
        assert loci == 6  # the headline models keep the largest group


def test_larger_models_get_smaller_groups():
    sizes = [_plan(immodel.build(_ladder(P)))[1] for P in (3, 4, 5)]
    assert sizes[0] >= sizes[1] >= sizes[2]
    assert sizes[2] < 6


def test_group_choice_is_maximal():
    """One more locus per group would exceed 64 KiB (or the group cap of 6):
    the planner shrinks groups only as far as the limit needs."""
    for P in (4, 5):
        model = immodel.build(_ladder(P))
        rc, loci, lds = _plan(model)
        assert rc == L.IMA_OK
        if loci < 6:
            # LDS grows with the group: 2^D scenario slots per parameter
            # plus D rows of records, so D + 1 must not fit
            per_locus_rows = 6 * (3 * P * P + 2 * P ** 3 + 1) * 8
            assert lds + per_locus_rows > 65536 or lds * 2 > 65536


def test_plan_rejects_bad_sizes():
    lib = L.load()
    loci, lds = C.c_int(), C.c_int64()
    assert lib.ima_mc3_prior_plan(0, 1, 1, 0, 0, C.byref(loci), C.byref(lds)) == L.ERR_ARG
    assert lib.ima_mc3_prior_plan(11, 1, 1, 0, 0, C.byref(loci), C.byref(lds)) == L.ERR_ARG


def _popmig_plan(rows, nx, expo):
    chunks, per, work = C.c_int(), C.c_int(), C.c_int64()
    assert L.load().ima_lmode_popmig_plan(rows, nx, expo, C.byref(chunks), C.byref(per),
                                          C.byref(work)) == L.IMA_OK
    return chunks.value, per.value, work.value


@pytest.mark.parametrize("expo", [0, 1])
@pytest.mark.parametrize("nx", [1, 255, 256, 4096])
def test_popmig_partials_fit_their_work_area(nx, expo):
    around = [n + d for n in (49152, 65536, 131072, 1000000, 3000000, 2 * 10 ** 9)
              for d in (-1, 0, 1, 4097)]
    for rows in list(range(1, 40001)) + around:
        chunks, per, work = _popmig_plan(rows, nx, expo)
        assert (chunks - 1) * per < rows <= chunks * per and chunks <= 1024
        assert work >= nx * chunks * (2 if expo else 1) * 8


@pytest.mark.parametrize("expo", [0, 1])
@pytest.mark.parametrize("rows", [1, 64, 20000, 65536, 65537, 1000000, 2 * 10 ** 9])
def test_popmig_work_area_is_bounded(rows, expo):
    """However many points: a caller with 10^8 of them needs no more."""
    for nx in (4096, 10 ** 5, 10 ** 8, 2 ** 31 - 1):
        chunks, _, work = _popmig_plan(rows, nx, expo)
        per = chunks * (2 if expo else 1) * 8
        assert min(nx, 4096) * per <= work <= 64 << 20


def test_popmig_plan_rejects_bad_sizes():
    a, b, w = C.c_int(), C.c_int(), C.c_int64()
    lib = L.load()
    assert lib.ima_lmode_popmig_plan(0, 1, 0, C.byref(a), C.byref(b), C.byref(w)) == L.ERR_ARG
    assert lib.ima_lmode_popmig_plan(1, -1, 0, C.byref(a), C.byref(b), C.byref(w)) == L.ERR_ARG
    assert lib.ima_lmode_popmig_plan(1, 1, 0, None, C.byref(b), C.byref(w)) == L.ERR_ARG
