"""Block tiles with two groups of wavefronts that share K (mmt4d_mfma_kernels.h, two_groups): the 128x128 tile of 16-bit operands
with either output, of int8 with row pieces of every size but two bytes and of an int4 rhs, and the 64x128 tile of an int4 rhs. From
44 chunks of 64 bytes on, an even and an odd number of them, K ending at every place of a chunk that row pieces leave, either
group's first chunk being the one that is cut or none; ragged last tiles. That the problems do take two groups, which the
kernel's name does not say, is checked in test_block_kernel_forms_on_host.py. Tolerances as in test_gpu_big_tiles: integers exact.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, F16, BF16, S8S4 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32, abi.MMT4D_TYPE_S8S4S32
F16_OUT16, BF16_OUT16 = abi.MMT4D_TYPE_F16F16F16, abi.MMT4D_TYPE_BF16BF16BF16

SIXTEEN_BIT = [(BF16, 16, 16, 16), (BF16, 8, 8, 4), (F16, 16, 16, 8), (F16, 4, 8, 2), (BF16, 1, 16, 16), (BF16_OUT16, 16, 16, 16),
               (BF16_OUT16, 8, 8, 4), (F16_OUT16, 16, 16, 16), (F16_OUT16, 8, 16, 2), (F16, 8, 8, 4), (F16, 16, 16, 32)]
EIGHT_BIT = [(8, 8, 1), (16, 16, 1), (8, 16, 1), (8, 8, 4), (16, 16, 4), (4, 16, 4), (8, 8, 8), (16, 4, 8), (16, 16, 16), (16, 8, 32),
             (16, 16, 64), (1, 16, 64), (1, 16, 16)]
FOUR_BIT = [(16, 16, 32), (8, 4, 64), (1, 16, 32)]


def sixteen_bit_problems(flags, M0, N0, K0):
    """Tiles and options of the calls: (M, N, K, options of run_case)."""
    ks = 32 // K0  # k steps of a chunk
    for n, (rows, cols) in enumerate([(1000, 2064), (640, 4000)]):
        for K in (64 * ks, 65 * ks, 66 * ks - 1, 66 * ks + 1, 71 * ks + ks // 2, 113 * ks):
            yield -(-rows // M0), cols // N0, K, dict(out_pad=4 if n else 0, accumulate=K % 2 == 0, seed=n)


def eight_bit_problems(M0, N0, K0):
    ks = 64 // K0
    for n, (rows, cols) in enumerate([(1000, 2064), (640, 4000)]):
        for K in (44 * ks, 45 * ks, 48 * ks - 1 - n, 48 * ks + 1 + n, 51 * ks - ks // 2, 64 * ks - ks // 4, 65 * ks - ks // 4):
            # (tile rows a multiple of 16 bytes apart, as the direct-to-LDS kernel needs)
            pad = [-K * M0 * K0 % 16 + 64 * n, -K * N0 * K0 % 16 + 128 * n]
            yield -(-rows // M0), cols // N0, K, dict(lhs_pad=pad[0], rhs_pad=pad[1], out_pad=4 * n, accumulate=K % 2 == 1, seed=n)


def four_bit_problems(M0, N0, K0, sizes):
    ks = 64 // K0
    for n, (rows, cols) in enumerate(sizes):
        for K in (64 * ks, 65 * ks, 66 * ks - (K0 == 32), 66 * ks + (K0 == 32), 129 * ks):
            yield -(-rows // M0), cols // N0, K, dict(accumulate=n == 1, seed=n)


TALL, WIDE = [(1000, 2064), (2672, 784)], [(512, 4000), (248, 7800)]  # 128x128 and 64x128 tiles of an int4 rhs


@pytest.mark.parametrize("flags,M0,N0,K0", SIXTEEN_BIT)
def test_16_bit_operands(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    for M, N, K, options in sixteen_bit_problems(flags, M0, N0, K0):
        run_case(gpu_lib, flags, M, N, K, M0, N0, K0, "mmt4d_mfma_128x128", **options)


@pytest.mark.parametrize("M0,N0,K0", EIGHT_BIT)
def test_8_bit_operands(gpu_lib, M0, N0, K0):  # noqa: F811
    for M, N, K, options in eight_bit_problems(M0, N0, K0):
        run_case(gpu_lib, S8, M, N, K, M0, N0, K0, "mmt4d_mfma_128x128", **options)


@pytest.mark.parametrize("M0,N0,K0", FOUR_BIT)
@pytest.mark.parametrize("sizes,tile", [(WIDE, "64x128"), (TALL, "128x128")], ids=["64x128", "128x128"])
def test_four_bit_rhs(gpu_lib, M0, N0, K0, sizes, tile):  # noqa: F811
    for M, N, K, options in four_bit_problems(M0, N0, K0, sizes):
        run_case(gpu_lib, S8S4, M, N, K, M0, N0, K0, "mmt4d_mfma_" + tile, **options)
