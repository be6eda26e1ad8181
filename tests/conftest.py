import ctypes as C
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")
    config.addinivalue_line("markers", "slow: long CPU sweep, excluded from the default run")


@pytest.fixture(scope="session")
def oracle():
    from oracle import binding
    binding.build()
    return binding


@pytest.fixture(scope="session")
def hip():
    """The HIP backend over libferrite_hip.so (GPU tests only; it has no CPU path)."""
    from ferrite_amd.backend import HipBackend
    return HipBackend()


@pytest.fixture(scope="session")
def shim(tmp_path_factory):
    """Host build of the kernels' scalar numerics and of the rules that launches follow (numerics_host_shim.cpp)."""
    out = tmp_path_factory.mktemp("shim") / "libnumerics_shim.so"
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-o", str(out),
                           os.path.join(ROOT, "tests", "numerics_host_shim.cpp")])
    lib = C.CDLL(str(out))
    for f in ("shim_expf", "shim_sigmoid", "shim_e4m3_decode", "shim_e2m1_decode", "shim_ue8m0_decode"):
        getattr(lib, f).restype = C.c_float
    lib.shim_expf.argtypes = [C.c_float]
    lib.shim_sigmoid.argtypes = [C.c_float]
    lib.shim_swiglu.restype = C.c_float
    lib.shim_swiglu.argtypes = [C.c_float] * 3
    lib.shim_e4m3_encode.argtypes = [C.c_float]
    lib.shim_block_scale_e8m0.argtypes = [C.c_float]
    lib.shim_e4m3_decode.argtypes = [C.c_uint]
    lib.shim_e2m1_decode.argtypes = [C.c_uint]
    lib.shim_ue8m0_decode.argtypes = [C.c_uint]
    lib.shim_expf_many.argtypes = [C.c_void_p, C.c_void_p, C.c_long]
    lib.shim_stream_raise.argtypes = [C.POINTER(C.c_int), C.c_int, C.c_int]
    lib.shim_stream_blocks.argtypes = [C.c_int, C.POINTER(C.c_int)]
    lib.shim_stream_cover.argtypes = [C.c_int, C.c_int, C.c_void_p]
    return lib
