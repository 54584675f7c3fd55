"""The 128x128 tile of 16-bit operands and the 64x128 tile of an int4 rhs with two groups of wavefronts that share K
(mmt4d_mfma_kernels.h, two_groups): from 64 chunks of 64 bytes on, an even and an odd number of them, K ending at every place of
a chunk that row pieces leave, either group's first chunk being the one that is cut or none; ragged last tiles; both output types.
Tolerances as in test_gpu_big_tiles: integers exact.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

F16, BF16, S8S4 = abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32, abi.MMT4D_TYPE_S8S4S32
BF16_OUT16 = abi.MMT4D_TYPE_BF16BF16BF16


@pytest.mark.parametrize("flags,M0,N0,K0", [(BF16, 16, 16, 16), (BF16, 8, 8, 4), (F16, 16, 16, 8), (F16, 4, 8, 2), (BF16, 1, 16, 16),
                                            (BF16_OUT16, 16, 16, 16), (BF16_OUT16, 8, 8, 4)])
def test_16_bit_operands(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    for n, (rows, cols) in enumerate([(1000, 2064), (640, 4000)]):
        ks = 32 // K0  # k steps of a chunk
        for K in (64 * ks, 65 * ks, 66 * ks - 1, 66 * ks + 1, 71 * ks + ks // 2, 113 * ks):
            run_case(gpu_lib, flags, -(-rows // M0), cols // N0, K, M0, N0, K0, "mmt4d_mfma_128x128", out_pad=4 if n else 0,
                     accumulate=K % 2 == 0, seed=n)


@pytest.mark.parametrize("M0,N0,K0", [(16, 16, 32), (8, 4, 64), (1, 16, 32)])
def test_four_bit_rhs(gpu_lib, M0, N0, K0):  # noqa: F811
    for n, (rows, cols) in enumerate([(512, 4000), (248, 7800)]):
        ks = 64 // K0
        for K in (64 * ks, 65 * ks, 66 * ks - (K0 == 32), 66 * ks + (K0 == 32), 129 * ks):
            run_case(gpu_lib, S8S4, -(-rows // M0), cols // N0, K, M0, N0, K0, "mmt4d_mfma_64x128", accumulate=n == 1, seed=n)
