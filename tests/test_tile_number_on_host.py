"""Which block tile a workgroup takes (tile_of_number, iree_amd/csrc/uk_device.h), by multiplications, against divisions: compiled
for the host, tests/host_checks/tile_number_check.hip.
"""
import os

from iree_amd import build as hip_build
from test_device_rounding_on_host import ROOT, _run


def test_tile_numbers(tmp_path):
    exe = str(tmp_path / "tile_number_check")
    _run([hip_build.HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-I" + hip_build.CSRC,
          os.path.join(ROOT, "tests", "host_checks", "tile_number_check.hip"), "-o", exe])
    out = _run([exe])
    assert ", 0 wrong" in out and int(out.split()[0]) > 1000000, out
