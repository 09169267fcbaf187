"""The fix-up list of the no-allocation path: with every surviving slot sent
through it (debug bit 0) it has room for 256 of each quartet type's; the
others are kept by every class, which changes nothing here, and reported."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
KTOL_ABS, KTOL_REL = 1e-10, 1e-11   # the parity bar


def test_noalloc_reports_slots_without_an_entry(capfd):
    from libgint_amd import driver as D, load
    from test_zz_no_alloc import Hip, _noalloc, _planned

    lib = load()
    hip = Hip()
    s, st, P, h = _planned(lib, D, dict(n_water=1, box_A=6.0, image_shells=1, np_max=3, seed=2))
    K = []
    for debug in (0, 1):
        lib.libgint_amd_set_debug(h, debug)
        rc, k = _noalloc(lib, hip, s, h, P)
        assert rc == 0
        K.append(k)
        said = capfd.readouterr().err
        print("debug", debug, "max|K|", np.max(np.abs(k)), said)
        assert ("beyond the fix-up list" in said) == (debug == 1)
    lib.libgint_amd_destroy_handle(h)
    assert np.max(np.abs(K[0])) > 0
    assert np.max(np.abs(K[0] - K[1])) <= KTOL_ABS + KTOL_REL * np.max(np.abs(K[0]))
