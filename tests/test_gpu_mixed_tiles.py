"""The single-precision tiles of the matrix-core contraction (k_eco) in plans
that reach them: rows long enough for the rule (96 primitive quartets per row
of a type), and shorter ones with that kernel forced (debug bit 3).

Every set quartet is routed (a tau beyond all bounds), and how far K moves is
held against the oracle with the factors of the same classes' contraction
rounded to single precision: 2 ulps of 2^-24 a product, on the GPU up to 18
(16 products summed in single precision).  So no more than 10 times as far,
and at least a tenth: in FP64 runs K moves by 1e-9 of that, and tiles put
together wrongly move it by the whole."""
import ctypes as C

import os
import subprocess

import numpy as np
import pytest

from helpers import ROOT, oracle

pytestmark = pytest.mark.gpu
KTOL_ABS, KTOL_REL = 1e-10, 1e-11

CASES = {
    "long_rows": (dict(n_water=1, n_tm=1, box_A=5.0, np_min=4, np_max=4, np_tm=5, seed=31), 0),
    "forced": (dict(n_water=1, n_tm=1, box_A=6.0, image_shells=1, np_max=2, np_tm=3, seed=31), 8),
}


@pytest.fixture(scope="module")
def rounded(tmp_path_factory):
    """the oracle with the contraction of classes of at least 8 contractions in single precision"""
    import oracle as O

    with open(os.path.join(ROOT, "oracle", "oracle.c")) as f:
        src = f.read()
    line = "dstk[j] += Kp * AC0[j];"
    assert src.count(line) == 1
    d = str(tmp_path_factory.mktemp("oracle"))
    with open(os.path.join(d, "oracle.c"), "w") as f:
        f.write(src.replace(line, "dstk[j] += nlabcd >= 8 ? (double)((float)Kp * (float)AC0[j]) : Kp * AC0[j];"))
    so = os.path.join(d, "liboracle.so")
    subprocess.run(["gcc", "-O2", "-fPIC", "-shared", "-std=c99", "-fopenmp", "-ffp-contract=off", "-w",
                    "-I" + os.path.join(ROOT, "oracle"), "-o", so, os.path.join(d, "oracle.c"), "-lm"], check=True)
    lib = C.CDLL(so)
    for n, (res, args) in O.SIG.items():
        f = getattr(lib, n)
        f.restype, f.argtypes = res, args
    return lib


@pytest.mark.parametrize("name", list(CASES))
def test_single_precision_tiles(name, rounded):
    from libgint_amd import driver as D, load

    lib, o = load(), oracle()
    cfg, debug = CASES[name]
    s = D.System(**cfg)
    st = s.record()
    P = s.P()
    Ko, ho = D.kbuild(o, "oracle_", s, st, P=P)
    o.oracle_destroy_handle(ho)
    Kr, hr = D.kbuild(rounded, "oracle_", s, st, P=P)
    rounded.oracle_destroy_handle(hr)
    kmax, far = np.max(np.abs(Ko)), np.max(np.abs(Kr - Ko))
    h, table = D.setup_handle(lib, "libgint_", s, P=P, debug=debug)
    lib.libgint_amd_plan_begin(h)
    st.replay(table, h)
    lib.libgint_amd_plan_end(h)

    def k():
        lib.libgint_set_P(h, D._ptr(P), s.P_size)
        lib.libgint_amd_plan_execute(h)
        K = np.zeros(s.P_size)
        lib.libgint_get_K(h, D._ptr(K))
        return K

    tune, info = (C.c_double * 5)(), (C.c_double * 4)()
    lib.libgint_amd_tune_info(h, tune)
    K64 = [k(), k()]
    lib.libgint_amd_set_mixed_precision(h, 1e300)
    K64.append(k())   # the calibration
    for K in K64:
        assert np.max(np.abs(K - Ko)) <= KTOL_ABS + KTOL_REL * kmax
    for _ in range(3):
        K = k()
        lib.libgint_amd_mixed_info(h, info)
        moved = np.max(np.abs(K - K64[0]))
        print(name, "classes on k_eco", tune[3], "flagged", info[2], "of", info[3], "max|K|", kmax, "moved", moved,
              "oracle", far)
        assert info[2] == info[3] and (debug or tune[3] > 0)
        assert 0.1 * far <= moved <= 10 * far
    lib.libgint_amd_destroy_handle(h)
