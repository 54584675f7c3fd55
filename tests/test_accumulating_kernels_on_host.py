"""Block kernels for calls that accumulate and for those that do not, on the CPU: which one a call takes (host_launches.py), and, from
the built library's kernel descriptions, that the registers of a plain one leave room for the workgroups that the LDS has room for."""
import os
import re
import struct
import subprocess

import pytest

from iree_amd import abi
from iree_amd import build as hip_build
from host_launches import recorder  # noqa: F401

READELF = os.path.join(os.path.dirname(hip_build.CLANG), "llvm-readelf")
LDS, REGISTERS = 160 * 1024, 512  # of a compute unit; of a lane of a SIMD, shared by the wavefronts on it
NAME = re.compile(r"mmt4d_mfma_direct_kernelILi(\d)ELb(\d)ELb(\d)ELi(\d+)ELi(\d)ELi(\d)ELi(\d+)ELi(\d)ELi(\d)ELi(\d)E")
NEVER, ALWAYS, ASKED = 0, 1, 2


def registers(path, out):
    """Kernel symbol -> vector registers of a lane, of every gfx950 code object in the library."""
    data, found, at = open(path, "rb").read(), {}, 0
    while (at := data.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if b"gfx950" in target and size:
                out.write_bytes(data[at + offset:at + offset + size])
                notes = subprocess.run([READELF, "--notes", str(out)], stdout=subprocess.PIPE, text=True, check=True).stdout
                for kernel in re.split(r"\n  - ", notes)[1:]:
                    symbol, count = re.search(r"\.symbol:\s+'?(\S+?)\.kd", kernel), re.search(r"\.vgpr_count:\s+(\d+)", kernel)
                    if symbol and count:  # (the notes' other lists)
                        found[symbol[1]] = int(count[1])
        at += 24
    return found


def test_registers_leave_room_for_the_workgroups_that_the_lds_holds(tmp_path):
    if not os.path.exists(hip_build.LIB_PATH):
        hip_build.build()
    plain = 0
    for symbol, count in registers(hip_build.LIB_PATH, tmp_path / "object").items():
        m = NAME.search(symbol)
        if not m or int(m[10]) != NEVER:
            continue
        rhs_i4, am, bn, stages, groups = int(m[2]), int(m[5]), int(m[6]), int(m[7]), int(m[9])
        workgroups = LDS // (groups * stages * 16 * (256 * am + (128 if rhs_i4 else 256) * bn))
        # (Four wavefronts, one a SIMD, of a group; registers come eight at a time.)
        assert REGISTERS // (-(-count // 8) * 8) >= workgroups * groups, (symbol, count, workgroups)
        plain += 1
    assert plain >= 100


# Tiles; M0, N0, K0 of 16-, 8-, 4- and 2-byte row pieces; the last has pairs of fragments, whose kernels are for calls of both kinds.
@pytest.mark.parametrize("flags,M0,N0,K0,pairs", [
    (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 16, False), (abi.MMT4D_TYPE_S8S4S32, 16, 16, 32, False), (abi.MMT4D_TYPE_F32F32F32, 16, 16, 4, False),
    (abi.MMT4D_TYPE_F16F16F16 | abi.MMT4D_SKIP_INTERMEDIATE_ROUNDINGS, 16, 16, 4, False), (abi.MMT4D_TYPE_S8S8S32, 8, 8, 4, False),
    (abi.MMT4D_TYPE_S8S8S32, 16, 16, 2, True), (abi.MMT4D_TYPE_F16F16F32, 16, 16, 1, True)])
def test_which_one_a_call_takes(recorder, flags, M0, N0, K0, pairs):  # noqa: F811
    element = {abi.MMT4D_TYPE_F32F32F32: 4, abi.MMT4D_TYPE_S8S8S32: 1, abi.MMT4D_TYPE_S8S4S32: 1}.get(flags, 2)
    for rows, cols, chunks in [(2048, 2048, 40), (1040, 12080, 9), (512, 14336, 44), (2064, 5136, 33)]:
        k = 64 * chunks // element - K0  # (a cut chunk, where 256x256 tiles have no tail of their own)
        kinds = []
        for accumulate in (0, abi.MMT4D_ACCUMULATE):
            m = NAME.search(recorder.mmt4d(flags | accumulate, -(-rows // M0), -(-cols // N0), k // K0, M0, N0, K0)[0])
            assert m, (rows, cols, k)
            kinds.append(int(m[10]))
        assert kinds == ([ASKED, ASKED] if pairs else [NEVER, ALWAYS]), (rows, cols, k)
