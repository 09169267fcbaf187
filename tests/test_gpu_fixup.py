"""The fix-up list of the no-allocation path: with every surviving slot sent
through it (debug bit 0) it has room for 256 of each quartet type's; the
others are kept by every class, which changes nothing here, and reported."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
KTOL_ABS, KTOL_REL = 1e-10, 1e-11   # the parity bar


def test_noalloc_reports_slots_without_an_entry(capfd):
    import torch

    from libgint_amd import driver as D, load

    lib = load()
    s = D.System(n_water=1, box_A=6.0, image_shells=1, np_max=3, seed=2)
    st = s.record()
    P = s.P()
    h, table = D.setup_handle(lib, "libgint_", s, P=P)
    lib.libgint_amd_plan_begin(h)
    st.replay(table, h)
    lib.libgint_amd_plan_end(h)
    dP = torch.from_numpy(P).cuda()
    K = []
    for debug in (0, 1):
        dK = torch.zeros_like(dP)
        torch.cuda.synchronize()
        lib.libgint_amd_set_debug(h, debug)
        assert lib.libgint_amd_plan_execute_noalloc(h, dP.data_ptr(), None, dK.data_ptr(), None, s.P_size) == 0
        lib.libgint_amd_synchronize(h)
        K.append(dK.cpu().numpy())
        said = capfd.readouterr().err
        print("debug", debug, "max|K|", np.max(np.abs(K[-1])), said)
        assert ("beyond the fix-up list" in said) == (debug == 1)
    lib.libgint_amd_destroy_handle(h)
    assert np.max(np.abs(K[0])) > 0
    assert np.max(np.abs(K[0] - K[1])) <= KTOL_ABS + KTOL_REL * np.max(np.abs(K[0]))
