"""The quartet kernel (blocks -> contraction, HRR, spherical transform, K) at
the edges of its tiles and windows, against the oracle: rows of 1 to 81
primitive quartets (its windows hold 16, in steps of 4), every kind of K
layout record, one and two spins, shell structures whose sides are one tile,
several tiles and, with f shells, tiles of a single contraction; the
contraction in the kernel itself and in its own kernel (debug bits 4 and 3).
Bar: 1e-10 Ha + 1e-11 max|K|, the K-build's conditioning (test_conditioning)."""
import functools

import numpy as np
import pytest

from helpers import oracle

pytestmark = pytest.mark.gpu
KTOL_ABS, KTOL_REL = 1e-10, 1e-11

CASES = {
    "np1": dict(n_water=2, box_A=7.0, image_shells=1, np_max=1, seed=4),
    "np2_one_cell": dict(n_water=2, box_A=5.0, np_min=2, np_max=2, seed=3),
    "np3_calls_reordered": dict(n_water=2, box_A=5.0, np_min=3, np_max=3, seed=6, ks_mix=1),
    "small_basis": dict(n_water=3, box_A=6.0, basis=1, np_min=2, np_max=3, seed=8),
    "f_basis": dict(n_water=1, box_A=5.0, basis=4, np_min=2, np_max=3, seed=2),
    "spdf_centre": dict(n_water=1, n_tm=1, box_A=6.0, np_max=2, np_tm=3, seed=9),
}


@pytest.mark.parametrize("spins", [1, 2])
@pytest.mark.parametrize("debug", [8, 16])
@pytest.mark.parametrize("name", list(CASES))
def test_tiles_and_windows(name, debug, spins):
    from libgint_amd import driver as D, load

    lib, o = load(), oracle()
    s = D.System(**CASES[name])
    st = s.record()
    P = s.P()
    kw = dict(P=P)
    if spins == 2:
        kw["Pb"] = P[::-1].copy()
    Ko, ho = D.kbuild(o, "oracle_", s, st, **kw)
    o.oracle_destroy_handle(ho)
    for plan in (False, True):
        K, h = D.kbuild(lib, "libgint_", s, st, plan=plan, debug=debug, **kw)
        lib.libgint_amd_destroy_handle(h)
        for a, b in zip(np.atleast_2d(K), np.atleast_2d(Ko)):
            err, kmax = np.max(np.abs(a - b)), np.max(np.abs(b))
            print(name, "debug", debug, "plan", plan, "sets", st.n_sets, "prm", st.n_prm, "max|K|", kmax, "max|dK|", err)
            assert kmax > 0 and err <= KTOL_ABS + KTOL_REL * kmax


# launch sets: the chunks of many quartet types from one launch per kernel, at
# most 64 chunks in a set and within half the memory budget
LAUNCH_SETS = {
    "many_types": (dict(n_water=4, n_tm=2, box_A=8.0, np_max=2, np_tm=2, seed=13), 4096),
    # set quartets of 1296 primitive quartets, in parts; of one and many rows, with long rows contracted by k_eco
    "parts_one_row": (dict(n_water=2, box_A=5.0, np_min=6, np_max=6, seed=15), 4096),
    "parts_many_rows": (dict(n_water=2, box_A=6.0, image_shells=1, np_min=6, np_max=6, basis=1, zmin=0.3, seed=16), 4096),
    "parts_spdf": (dict(n_water=1, n_tm=1, box_A=5.0, np_min=3, np_max=3, np_tm=7, seed=17), 4096),
    "several_sets_by_memory": (dict(n_water=5, box_A=7.0, np_min=3, np_max=3, seed=14), 64),
}


@functools.cache
def launch_set_reference(name):
    from libgint_amd import driver as D

    o = oracle()
    s = D.System(**LAUNCH_SETS[name][0])
    st = s.record()
    P = s.P()
    Ko, ho = D.kbuild(o, "oracle_", s, st, P=P)
    o.oracle_destroy_handle(ho)
    return s, st, P, Ko


@pytest.mark.parametrize("flags", [0, 1, 2])
@pytest.mark.parametrize("name", list(LAUNCH_SETS))
def test_launch_sets(name, flags):
    """flags: every surviving slot through the fix-up (1), one stream (2)"""
    from libgint_amd import driver as D, load

    lib = load()
    mib = LAUNCH_SETS[name][1]
    s, st, P, Ko = launch_set_reference(name)
    kmax = np.max(np.abs(Ko))
    for plan in (False, True):
        K, h = D.kbuild(lib, "libgint_", s, st, P=P, plan=plan, debug=flags, max_mem_mib=mib)
        lib.libgint_amd_destroy_handle(h)
        err = np.max(np.abs(K - Ko))
        print(name, "flags", flags, "plan", plan, "sets", st.n_sets, "prm", st.n_prm, "max|K|", kmax, "max|dK|", err)
        assert kmax > 0 and err <= KTOL_ABS + KTOL_REL * kmax
