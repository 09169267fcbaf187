"""The host engine (queues, plans, launch lists, request loop) built with a
HIP runtime over host memory and launchers that do no work (tests/host), for
tests of the host side on a CPU."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

from helpers import ROOT

CSRC = os.path.join(ROOT, "libgint_amd", "csrc")
HERE = os.path.join(ROOT, "tests", "host")
FLAGS = ["-g", "-O1", "-std=c++17", "-fPIC", "-fopenmp", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
         "-I/opt/rocm/include", "-I" + CSRC]
SRC = [os.path.join(CSRC, f) for f in ("engine.cpp", "abi.cpp", "plan.cpp", "boys_table.cpp", "c0_file.cpp", "server.cpp")]


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


def objects(out):
    """the engine's and the stub's objects in the folder `out`"""
    objs = [os.path.join(out, os.path.basename(f) + ".o") for f in SRC + ["stub.cpp"]]
    if not all(os.path.exists(o) for o in objs):
        with ThreadPoolExecutor(max_workers=4) as ex:
            list(ex.map(lambda x: _run(["g++"] + FLAGS + ["-c", x[0], "-o", x[1]]),
                        zip(SRC + [os.path.join(HERE, "stub.cpp")], objs)))
    return objs


def program(out, source):
    """the program tests/host/`source` linked with them"""
    exe = os.path.join(out, source + ".exe")
    _run(["g++"] + FLAGS + [os.path.join(HERE, source)] + objects(out) + ["-o", exe, "-lpthread", "-ldl"])
    return exe


def library(out):
    """them as a library, with the product's entry points declared"""
    import ctypes as C

    from libgint_amd import ABI

    so = os.path.join(out, "libgint_host.so")
    if not os.path.exists(so):
        _run(["g++", "-shared", "-fopenmp"] + objects(out) + ["-o", so])
    lib = C.CDLL(so)
    for name, (res, args) in ABI.items():
        f = getattr(lib, name)
        f.restype, f.argtypes = res, args
    return lib
