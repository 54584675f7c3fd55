"""Which mmt4d kernel the host picks, on the CPU (host_launches.py): for problems that were timed with every kernel, the one
picked is within 8 % of the best, in the geometric mean of operands that the last-level cache holds and operands from HBM."""
import math
import re

import pytest

from iree_amd import abi
from host_launches import recorder  # noqa: F401

LAYOUTS = {"bf16": (abi.MMT4D_TYPE_BF16BF16F32, 16, 16, 16), "s8": (abi.MMT4D_TYPE_S8S8S32, 16, 16, 64),
           "s8s4": (abi.MMT4D_TYPE_S8S4S32, 16, 16, 32), "f16, 2-byte pieces": (abi.MMT4D_TYPE_F16F16F32, 16, 16, 1),
           "s8, 4-byte pieces": (abi.MMT4D_TYPE_S8S8S32, 8, 8, 4), "bf16, 8-byte pieces": (abi.MMT4D_TYPE_BF16BF16F32, 8, 8, 4),
           "s8, 2-byte pieces": (abi.MMT4D_TYPE_S8S8S32, 16, 16, 2), "f32": (abi.MMT4D_TYPE_F32F32F32, 16, 16, 4)}

# Microseconds with operands held by the cache (150 MB in turn) and from HBM (640 MB in turn): the tiles of the kernel that
# splits K over wavefronts, and the block kernel that the problem would take.
TIMES = [
    ("bf16", 32, 11008, 2048, {"32x64": (9.8, 12.5), "64x64": (10.0, 12.8), "16x32": (10.4, 13.8), "block": (11.9, 13.2)}),
    ("bf16", 64, 4096, 4096, {"32x32": (9.2, 13.1), "16x32": (11.2, 16.0), "32x64": (11.0, 16.5), "block": (19.7, 21.0)}),
    ("bf16", 96, 14336, 4096, {"block": (23.9, 32.6), "64x64": (26.6, 38.4), "32x64": (27.5, 40.7)}),
    ("bf16", 512, 4096, 4096, {"block": (24.5, 30.0), "64x64": (26.4, 35.1), "64x32": (32.1, 42.4)}),
    ("s8", 64, 14336, 4096, {"64x64": (14.2, 14.7), "block": (12.8, 16.5), "32x64": (14.7, 19.3)}),
    ("s8", 128, 4096, 14336, {"32x64": (22.2, 26.9), "64x32": (22.1, 27.3), "32x32": (27.8, 33.1), "block": (32.0, 35.9)}),
    ("s8s4", 32, 28672, 8192, {"32x64": (25.4, 26.1), "16x32": (24.1, 33.9), "64x64": (28.4, 28.8), "block": (27.2, 30.7)}),
    ("s8s4", 96, 14336, 4096, {"block": (16.2, 16.3), "64x64": (15.8, 17.9), "32x64": (16.2, 19.3)}),
    ("s8s4", 96, 11008, 2048, {"block": (10.2, 10.3), "32x64": (10.8, 11.8), "64x64": (10.4, 12.4)}),
    ("s8s4", 192, 8192, 4096, {"64x64": (15.3, 17.9), "block": (16.6, 16.7), "32x64": (16.6, 18.7)}),
    ("f16, 2-byte pieces", 64, 4096, 4096, {"32x32": (10.8, 13.9), "16x32": (13.3, 16.7), "64x32": (14.0, 17.5), "block": (37.6, 37.9)}),
    ("s8, 4-byte pieces", 128, 2048, 2048, {"32x32": (5.6, 5.9), "16x32": (6.1, 6.4), "32x64": (6.5, 6.9), "block": (7.8, 7.9)}),
    ("bf16, 8-byte pieces", 32, 14336, 4096, {"32x64": (20.5, 25.2), "block": (19.9, 26.0), "64x64": (21.8, 26.6)}),
    ("s8, 2-byte pieces", 256, 11008, 2048, {"block": (15.5, 17.6), "64x64": (21.2, 23.8), "64x32": (28.1, 31.4)}),
    ("f32", 64, 2048, 2048, {"16x32": (10.2, 10.8), "16x16": (12.2, 13.0), "32x32": (15.9, 16.7), "block": (37.4, 37.5)}),
]


def kernel_of(mangled):
    """"block", or the tile of the kernel that splits K over wavefronts."""
    m = re.search(r"mmt4d_wave_k_kernelILi\dELb\dELb\dELi\d+ELi(\d)ELi(\d)E", mangled)
    if m:
        return "%dx%d" % (16 * int(m[1]), 16 * int(m[2]))
    assert "mmt4d_mfma" in mangled, mangled
    return "block"


@pytest.mark.parametrize("layout,m,n,k,times", TIMES, ids=lambda v: "times" if isinstance(v, dict) else str(v))
def test_the_kernel_picked_is_among_the_best(recorder, layout, m, n, k, times):  # noqa: F811
    flags, M0, N0, K0 = LAYOUTS[layout]
    mangled, _ = recorder.mmt4d(flags, m // M0, n // N0, k // K0, M0, N0, K0)
    picked = kernel_of(mangled)
    assert picked in times, mangled
    mean = {name: math.sqrt(held * hbm) for name, (held, hbm) in times.items()}
    assert mean[picked] <= 1.08 * min(mean.values()), (picked, mean)
