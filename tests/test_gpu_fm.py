"""The kernel from primitive quartets to blocks at the edges of its units (up
to 16 primitive quartets per wavefront, the last one short), of its lists of
slots (64 at a time, cells 0 to 255) and of its survivors (24 or 16 at a
time), against the oracle.  Bar: 1e-10 Ha + 1e-11 max|K|, the K-build's
conditioning (test_conditioning)."""
import numpy as np
import pytest

from helpers import oracle

pytestmark = pytest.mark.gpu
KTOL_ABS, KTOL_REL = 1e-10, 1e-11

CASES = {
    "full_units_one_cell": (dict(n_water=8, box_A=7.0, np_min=3, np_max=3, seed=14), {}),
    "full_units_coulomb": (dict(n_water=7, box_A=7.0, np_min=3, np_max=3, seed=15), dict(truncated=False)),
    "cells256": (dict(n_water=1, box_A=7.0, image_shells=3, np_max=2, zmin=0.6, seed=16), {}),
    "cells125_many_survivors": (dict(n_water=1, box_A=5.0, image_shells=2, np_max=2, basis=1, zmin=0.3, seed=17), {}),
}


@pytest.mark.parametrize("name", list(CASES))
def test_units_slots_survivors(name):
    from libgint_amd import driver as D, load

    lib, o = load(), oracle()
    cfg, kw = CASES[name]
    s = D.System(**cfg)
    st = s.record()
    P = s.P()
    Ko, ho = D.kbuild(o, "oracle_", s, st, P=P, **kw)
    o.oracle_destroy_handle(ho)
    kmax = np.max(np.abs(Ko))
    for plan in (False, True):
        K, h = D.kbuild(lib, "libgint_", s, st, P=P, plan=plan, **kw)
        lib.libgint_amd_destroy_handle(h)
        err = np.max(np.abs(K - Ko))
        print(name, "plan", plan, "cells", s.Ng, "sets", st.n_sets, "prm", st.n_prm, "max|K|", kmax, "max|dK|", err)
        assert kmax > 0 and err <= KTOL_ABS + KTOL_REL * kmax
