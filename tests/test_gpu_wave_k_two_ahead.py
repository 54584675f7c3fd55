"""The 16x16 tiles of the kernel that splits K over wavefronts (mmt4d_wave_k_kernels.h) with three to nine 64-byte steps of K
a wavefront, and around the number of steps from where two are in flight ahead (48, for f32 and
4-byte pieces 32; int8 in 16-byte pieces never): wavefronts with equally many steps or not, and K that ends inside a step.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
5200 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, F16, BF16, F32 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32, abi.MMT4D_TYPE_F32F32F32


@pytest.mark.parametrize("flags,T0,K0,e,two_from", [
    (BF16, 16, 16, 2, 48), (F16, 16, 16, 2, 48), (BF16, 16, 2, 2, 32), (F16, 16, 1, 2, 48), (S8, 16, 2, 1, 48), (S8, 8, 8, 1, 48),
    (S8, 16, 16, 1, 64), (F32, 16, 4, 4, 32), (F32, 16, 1, 4, 32), (F32, 16, 2, 4, 32)])
def test_steps(gpu_lib, flags, T0, K0, e, two_from):  # noqa: F811
    ksteps = 64 // (K0 * e)
    around = [two_from + d for d in (-2, -1, 0, 1, 7, 8, 9, 17, 40)]
    for n, steps in enumerate([31, 32, 33, 39, 40, 41, 47, 48, 55, 56, 57, 72, 119, 120, 128] + around):
        for rest in {0, ksteps // 4, ksteps - 1}:
            run_case(gpu_lib, flags, 48 // T0, 240 // T0, steps * ksteps + rest, T0, T0, K0, "mmt4d_mfma_wave_k_16x16",
                     accumulate=n % 3 == 1, seed=n)
