"""The library's host code on the CPU with a HIP runtime that notes launches instead of making them
(host_checks/recording_runtime.cpp): which kernel, grid and LDS size a call asks for."""
import concurrent.futures
import ctypes as C
import os
import subprocess

import pytest

from iree_amd import abi
from iree_amd import build as hip_build

RUNTIME = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_checks", "recording_runtime.cpp")


def _run(cmd):
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, "%s\n%s" % (" ".join(cmd), r.stdout[-4000:])
    return r.stdout


def build(out_dir):
    flags = [f for f in hip_build.COMMON_FLAGS if f != "-O3"] + ["-O1", "--offload-host-only", "-I" + hip_build.CSRC]

    def host_object(src):
        obj = os.path.join(out_dir, os.path.basename(src) + ".o")
        _run([hip_build.HIPCC] + flags + (["-fvisibility=default"] if src == RUNTIME else []) + ["-c", src, "-o", obj])
        return obj

    # (multi_mma.hip is left out: its kernels need the device bitcode, and its entry point is not a microkernel call.)
    sources = [os.path.join(hip_build.CSRC, s) for s in hip_build.sources() if s != "multi_mma.hip"] + [RUNTIME]
    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as pool:
        objs = list(pool.map(host_object, sources))
    # The device code that the objects would register, which nothing looks at.
    undefined = sorted({w for o in objs for l in _run(["nm", "-u", o]).splitlines() for w in l.split()[1:]
                        if w.startswith("__hip_fatbin")})
    rest = os.path.join(out_dir, "rest.cpp")
    with open(rest, "w") as f:
        f.write("".join('extern "C" const char %s[1] = {0};\n' % u for u in undefined))
        f.write('#include "uk_internal.h"\nhipError_t uk::launch_multi_mma_i8(const void*, const void*, void*, int64_t, int64_t, '
                'int32_t, int, int, int, int, int, hipStream_t) { return hipErrorInvalidValue; }\n')
    lib = os.path.join(out_dir, "librecording.so")
    _run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + hip_build.CSRC,
          "-Wl,-Bsymbolic", rest] + objs + ["-o", lib, "-lpthread"])
    return lib


class Recorder:
    def __init__(self, path):
        self.lib = C.CDLL(path)
        self.lib.recorded_kernel.restype = self.lib.iree_uk_mi355x_last_kernel.restype = C.c_char_p
        self.lib.recorded_lds.restype = C.c_size_t
        self.lib.iree_uk_mi355x_set_stream.argtypes = [C.c_void_p, C.c_int]

    def call(self, entry, params):
        """One call in the calling thread's asynchronous mode; the kernel's mangled name and the reported one."""
        self.lib.iree_uk_mi355x_set_stream(None, 1)
        self.lib.recorded_reset()
        getattr(self.lib, entry)(C.byref(params))
        return self.lib.recorded_kernel().decode(), self.lib.iree_uk_mi355x_last_kernel().decode()

    def mmt4d(self, flags, M, N, K, M0, N0, K0, lhs_pad=0, rhs_pad=0, out_pad=0, lhs=1 << 40, rhs=2 << 40, out=3 << 40):
        p = abi.Mmt4dParams()
        p.lhs_buffer, p.rhs_buffer, p.out_buffer = lhs, rhs, out
        p.lhs_stride0, p.rhs_stride0, p.out_stride0 = K * M0 * K0 + lhs_pad, K * N0 * K0 + rhs_pad, N * M0 * N0 + out_pad
        p.M, p.N, p.K, p.M0, p.N0, p.K0, p.flags = M, N, K, M0, N0, K0, flags
        return self.call("iree_uk_mmt4d_p", p)


@pytest.fixture(scope="session")
def recorder(tmp_path_factory):
    return Recorder(build(str(tmp_path_factory.mktemp("recording"))))
