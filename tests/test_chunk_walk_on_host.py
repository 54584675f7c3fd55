"""Where the direct-to-LDS kernel's steps load from and to (iree_amd/csrc/mmt4d_chunk_walk.h): compiled for the host and walked for every
number of chunks and every end of K, tests/host_checks/chunk_walk_check.hip.
"""
import os

from iree_amd import build as hip_build
from test_device_rounding_on_host import ROOT, _run


def test_chunk_walk(tmp_path):
    exe = str(tmp_path / "chunk_walk_check")
    _run([hip_build.HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-I" + hip_build.CSRC,
          os.path.join(ROOT, "tests", "host_checks", "chunk_walk_check.hip"), "-o", exe])
    out = _run([exe])
    assert ", 0 wrong" in out and int(out.split()[0]) > 10000, out
