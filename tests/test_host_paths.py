"""Host paths of the solver on the CPU: the host C++ linked with the device
objects of the last build over a HIP runtime of its own (native/fake_hip.cpp),
whose kernels do nothing and whose launches check their pointers.  Every
allocation of a call fails once; afterwards nothing may launch on memory that
is not live, and the problem has to work as before."""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

import pytest

from tmr_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
WRAP = "_ZN4tmrx6Forest27create_interpolation_deviceEPS0_RNS_9InterpCSREiPd"


@pytest.fixture(scope="module")
def fake_lib(tmp_path_factory):
    cpp, hip = build._sources()
    dev = [os.path.join(build.OUT_DIR, os.path.basename(s) + ".o") for s in hip]
    if not all(os.path.exists(o) for o in dev):
        pytest.skip("device objects missing (run the build first)")
    out = str(tmp_path_factory.mktemp("fake"))

    def compile_one(src):
        o = os.path.join(out, os.path.basename(src) + ".o")
        build._run(["g++"] + [f if f != "-O3" else "-O1" for f in build.CXX_FLAGS] +
                   ["-c", src, "-o", o])
        return o
    with ThreadPoolExecutor(max_workers=4) as ex:
        objs = list(ex.map(compile_one, cpp + [os.path.join(HERE, "native", "fake_hip.cpp")]))
    lib = os.path.join(out, "libtmrx_fake.so")
    build._run(["g++", "-shared", "-fPIC", "-Wl,-Bsymbolic", "-Wl,-z,defs",
                "-Wl,--wrap=" + WRAP, "-o", lib] + objs + dev)
    return lib


def _child(lib, *args):
    env = dict(os.environ, TMRX_LIB=lib,
               PYTHONPATH=ROOT + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, os.path.join(HERE, "native", "host_paths.py")] + list(args),
                       cwd=ROOT, env=env, capture_output=True, text=True, timeout=300)
    print(r.stdout[-2000:] + r.stderr[-2000:])
    assert r.returncode == 0


@pytest.mark.parametrize("call", [
    "solve", "FP64 solve", "three cases", "degree", "nodal design", "Galerkin", "SOR",
    "matrix cores", "tiling", "autotune", "filter"])
def test_failed_allocations(fake_lib, call):
    _child(fake_lib, call)


def test_default_tiles_fit_in_lds(fake_lib):
    _child(fake_lib, "LDS")
