"""libqiw's own objects linked with a HIP runtime that records launches (native/hip_stub.cpp):
the host code of the library (programs, plans, captures, device buffers) on the CPU."""
import collections
import ctypes as C
import glob
import os
import shutil
import subprocess
from unittest import mock

import pytest

from qiw import abi

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(HERE, "..", "qinchworm.jl_amd")
NAMES = ["kernels", "arcs", "flow", "host", "warp"]

Launch = collections.namedtuple("Launch", "name grid block lds args freed")


class Stub:
    """One context on the recording runtime."""

    def __init__(self, path):
        # beside a libqiw.so of the same process: names bound to this library's own copy
        with mock.patch.object(abi, "_lib", None), mock.patch.object(C, "RTLD_GLOBAL", C.RTLD_LOCAL):
            self.lib = abi.load_library(path)
            self.ctx = abi.Context()
        self.lib.stub_name.restype = C.c_char_p
        self.lib.stub_peak_bytes.restype = self.lib.stub_copies.restype = C.c_size_t

    def clear(self):
        self.lib.stub_clear()

    def launches(self, *names):
        """What has run since clear(), kernels with one of `names` in their names."""
        out = []
        for i in range(self.lib.stub_launches()):
            name = self.lib.stub_name(i).decode()
            if names and not any(n in name for n in names):
                continue
            shape, p = (C.c_int64 * 7)(), C.c_void_p()
            self.lib.stub_shape(i, shape)
            n = self.lib.stub_args(i, C.byref(p))
            out.append(Launch(name, tuple(shape[0:3]), tuple(shape[3:6]), shape[6], C.string_at(p, n) if n else b"",
                              self.lib.stub_freed_args(i)))
        return out


@pytest.fixture(scope="module")
def stub_path(tmp_path_factory):
    gxx, rocm = shutil.which("g++"), "/opt/rocm"
    if gxx is None or not os.path.isdir(os.path.join(rocm, "include", "hip")):
        pytest.skip("g++ or the HIP headers not available")
    objs = [os.path.join(PKG, "build", f"qiw_{n}.o") for n in NAMES]
    if not all(os.path.exists(o) for o in objs):
        subprocess.run(["make", "-j", "4", "-C", PKG], check=True)
    assert set(glob.glob(os.path.join(PKG, "build", "qiw_*.o"))) >= set(objs)
    so = str(tmp_path_factory.mktemp("stub") / "libqiw_stub.so")
    subprocess.run([gxx, "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-D__HIP_PLATFORM_AMD__", "-w",
                    "-I", os.path.join(rocm, "include"), "-I", os.path.join(PKG, "csrc"), "-I", os.path.join(HERE, "..", "include"),
                    os.path.join(HERE, "native", "hip_stub.cpp"), *objs, "-o", so, "-lpthread"], check=True)
    return so


@pytest.fixture
def stub(stub_path):
    s = Stub(stub_path)
    yield s
    s.ctx.close()
