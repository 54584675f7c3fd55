"""K that ends inside a 64-byte step on the 16x32 tiles of the kernel that splits K over wavefronts (mmt4d_wave_k_kernels.h),
whose operands pass through LDS (row pieces of 2, 4 and 8 bytes) and whose last step is loaded ahead of the others: none, one
and several whole steps a wavefront, every remainder of a k step.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
1100 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, F16, BF16 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32


@pytest.mark.parametrize("flags,T0,N0,K0,e,rows", [(F16, 8, 16, 1, 2, 8), (S8, 16, 16, 2, 1, 16), (S8, 8, 8, 8, 1, 16), (S8, 8, 8, 4, 1, 16),
                                                   (BF16, 8, 8, 4, 2, 16)])
def test_rest(gpu_lib, flags, T0, N0, K0, e, rows):  # noqa: F811
    ksteps = 64 // (K0 * e)
    for n, steps in enumerate([3, 7, 8, 9, 15, 16, 17, 24, 25, 33]):
        for rest in sorted({0, 1, 2, ksteps // 2, ksteps - 1}):
            run_case(gpu_lib, flags, rows // T0, 8192 // N0, steps * ksteps + rest, T0, N0, K0, "mmt4d_mfma_wave_k_16x32",
                     accumulate=n % 3 == 1, seed=n)
