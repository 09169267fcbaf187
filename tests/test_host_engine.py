"""The host engine without a GPU (tests/host): what a plan keeps while other
calls come in between, and the room that its launch sets have."""
import ctypes as C

import numpy as np
import pytest

import hostlib


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return hostlib.library(str(tmp_path_factory.mktemp("host")))


def _planned(lib, **kw):
    from libgint_amd import driver as D

    s = D.System(**kw)
    st = s.record()
    P = s.P()
    h, table = D.setup_handle(lib, "libgint_", s, P=P)
    lib.libgint_amd_plan_begin(h)
    st.replay(table, h)
    lib.libgint_amd_plan_end(h)
    return s, st, P, h, table


def test_graph_kept_over_streamed_work(lib):
    """a plan's captured graph serves its next execution also when set
    quartets were streamed through the handle in between"""
    from libgint_amd import driver as D

    s, st, P, h, table = _planned(lib, n_water=1, box_A=4.0, np_max=2, seed=2)
    K = np.zeros(s.P_size)
    info = (C.c_uint64 * 4)()
    for _ in range(3):
        lib.libgint_set_P(h, D._ptr(P), s.P_size)
        lib.libgint_amd_plan_execute(h)
        st.replay(table, h, 0, st.n_sets // 2)
        lib.libgint_get_K(h, D._ptr(K))
    lib.libgint_amd_graph_info(h, info)
    lib.libgint_amd_destroy_handle(h)
    assert list(info) == [1, 1, 3, 1]


def test_noalloc_after_new_lattice_vectors(lib):
    """plan_execute_noalloc refuses while new lattice vectors are not on the
    device, and takes the plan again once plan_execute has put them there"""
    from libgint_amd import driver as D

    s, st, P, h, table = _planned(lib, n_water=1, box_A=6.0, image_shells=1, np_max=2, seed=2)
    n = s.P_size
    dK = np.zeros(n)
    ptr = lambda a: a.ctypes.data  # noqa: E731

    def noalloc():
        return lib.libgint_amd_plan_execute_noalloc(h, ptr(P), None, ptr(dK), None, n)

    assert noalloc() == 0
    g = np.concatenate([s.neighs(), s.neighs() + 1.0])
    lib.libgint_set_neighs(h, D._ptr(g), 2 * s.Ng)
    assert noalloc() == -6
    lib.libgint_set_P(h, D._ptr(P), n)
    lib.libgint_amd_plan_execute(h)
    assert noalloc() == 0
    lib.libgint_amd_destroy_handle(h)


@pytest.mark.parametrize("noalloc,entries", [(False, 4096), (True, 256)])
def test_fixup_entries_of_every_chunk(lib, noalloc, entries):
    """every chunk of a launch set has its own entries of the fix-up list (a
    slot beyond them is kept by every class)"""
    from libgint_amd import driver as D

    s, st, P, h, table = _planned(lib, n_water=2, n_tm=1, box_A=6.0, np_max=2, np_tm=2, seed=2)
    if noalloc:
        dK = np.zeros(s.P_size)
        assert lib.libgint_amd_plan_execute_noalloc(h, P.ctypes.data, None, dK.ctypes.data, None, s.P_size) == 0
    else:
        lib.libgint_set_P(h, D._ptr(P), s.P_size)
        lib.libgint_amd_plan_execute(h)
    n = lib.stub_fix_chunks()
    rooms = [(lib.stub_fix_at(i), lib.stub_fix_cap(i)) for i in range(n)]
    lib.libgint_amd_destroy_handle(h)
    assert n > 1 and rooms == [(entries * i, entries) for i in range(n)]
