"""What the compiler makes of pack and unpack (pack_unpack_tiled.hip), read from the assembly.

The wait states behind the wide stores that pack writes through the caches (inline assembly): a vector instruction that
overwrites the registers of a store of more than 8 bytes has to stay clear of it, and the compiler, which sees to that
behind its own stores, does not look into assembly. What it keeps behind its own stores is read from a kernel in which the
next instruction is such a one, and every store of the package's assembly has to keep as much.

The loads of line-aligned unpack: 16 bytes each, however small the pieces are that go to LDS."""
import os
import re
import subprocess

import pytest

from iree_amd import build as hip_build

PROBE = r"""
#include <hip/hip_runtime.h>
typedef int v4i32 __attribute__((ext_vector_type(4)));
__global__ void overwrite(v4i32* p) {
  v4i32 v = {1, 2, 3, 4};
  asm volatile("; keep %0" : "+v"(v));
  __builtin_nontemporal_store(v, p);
  asm volatile("v_mov_b32 %0, 0 ; overwrite" : "+v"(v));
  asm volatile("; keep %0" : : "v"(v));
}
"""


def _assembly(source, out):
    r = subprocess.run([hip_build.HIPCC] + hip_build.COMMON_FLAGS + ["-S", "--cuda-device-only", source, "-o", out],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    return [l.split("//")[0].strip() for l in open(out)]


@pytest.fixture(scope="module")
def pack_assembly(tmp_path_factory):
    return _assembly(os.path.join(hip_build.CSRC, "pack_unpack_tiled.hip"), str(tmp_path_factory.mktemp("asm") / "pack.s"))


def _wait_states(lines):
    """Of a run of instructions: one each, s_nop n counts n + 1."""
    total = 0
    for l in lines:
        m = re.match(r"s_nop (\d+)", l)
        total += int(m.group(1)) + 1 if m else 1 if re.match(r"[sv]_", l) else 0
    return total


def test_every_store_in_assembly_keeps_the_compilers_distance(pack_assembly, tmp_path):
    src = tmp_path / "probe.hip"
    src.write_text(PROBE)
    probe = _assembly(str(src), str(tmp_path / "probe.s"))
    store = next(i for i, l in enumerate(probe) if l.startswith("global_store_dwordx4"))
    overwrite = next(i for i, l in enumerate(probe) if "overwrite" in l and l.startswith("v_mov"))
    needed = _wait_states(probe[store + 1:overwrite])
    assert needed >= 1, probe[store:overwrite + 1]

    text = pack_assembly
    stores = [i for i, l in enumerate(text) if re.match(r"global_store_dwordx4 .*\bsc1\b", l)]
    assert len(stores) >= 60
    short = [(i, text[i:i + 2]) for i in stores if _wait_states(text[i + 1:i + 2]) < needed]
    assert not short, (needed, len(short), short[:3])


def test_line_aligned_unpack_loads_whole_vectors(pack_assembly):
    # tiled_kernel<element bytes, 16, piece bytes, unpack, cache policy, line-aligned form>
    kernel, loads = None, {}
    for l in pack_assembly:
        m = re.match(r"_ZN2uk12_GLOBAL__N_112tiled_kernelILi(\d)ELi16ELi(\d+)ELb1ELi(\d)ELi([12])EEE\w*:", l)
        if m:
            kernel = m.groups()
            loads[kernel] = set()
        elif l.startswith("s_endpgm"):
            kernel = None
        elif kernel and l.startswith("global_load"):
            loads[kernel].add(l.split()[0])
    assert len(loads) == 28  # (three piece sizes of 4-byte elements and four of 2-byte ones, two policies and forms)
    assert all(v == {"global_load_dwordx4"} for v in loads.values()), {k: v for k, v in loads.items() if len(v) > 1}
