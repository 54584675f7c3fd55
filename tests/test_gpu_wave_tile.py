"""The kernel whose wavefronts multiply the whole of a large tile each (mmt4d_wave_tile.hip): 128x128 tiles of 16-bit operands with
either output, 64x128 tiles of an int4 rhs. Every remainder of the number of 64-byte chunks by the four
wavefronts and the two steps that one has in registers, K ending at every place of a chunk that row pieces leave, ragged last tiles. Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)):
sums of at most 4500 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order.
"""
import ctypes as C

import pytest
import torch

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, mm_params, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

F16, BF16, S8S4 = abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32, abi.MMT4D_TYPE_S8S4S32
F16_OUT16, BF16_OUT16 = abi.MMT4D_TYPE_F16F16F16, abi.MMT4D_TYPE_BF16BF16BF16

SIXTEEN_BIT = [(BF16, 16, 16, 16), (BF16, 16, 16, 8), (F16, 8, 16, 16), (F16, 4, 4, 8), (BF16_OUT16, 16, 8, 16), (F16_OUT16, 8, 4, 8)]
FOUR_BIT = [(16, 16), (8, 16), (16, 8), (4, 4)]  # M0, N0


def sixteen_bit_problems(M0, N0, K0):
    """Tiles and options of the calls: (M, N, K, options of run_case)."""
    ks = 32 // K0  # k steps of a chunk
    for n, (rows, cols, chunks) in enumerate([(1744, 1848, 64), (1552, 1952, 65), (3076, 960, 66), (424, 7804, 67), (1744, 2112, 68),
                                              (1552, 1940, 69), (404, 7804, 71), (3076, 960, 139)]):
        for rest in range(ks):
            yield (-(-rows // M0), -(-cols // N0), chunks * ks - rest,
                   dict(lhs_pad=64 * (n % 2), rhs_pad=16 * (n % 3), out_pad=4 * (n % 2), accumulate=n % 2 == 1, seed=n))


def four_bit_problems(M0, N0):
    for n, (rows, cols, chunks) in enumerate([(368, 2720, 30), (496, 2192, 45), (784, 1328, 37), (1424, 736, 44), (240, 4140, 52),
                                              (224, 4944, 41), (272, 3952, 103), (1824, 544, 39)]):
        for rest in (0, 1):  # k steps of 32 values
            yield (-(-rows // M0), -(-cols // N0), 2 * chunks - rest,
                   dict(lhs_pad=32 * (n % 2), rhs_pad=64 * (n % 3), out_pad=4 * (n % 2), accumulate=n % 2 == 1, seed=n))


@pytest.mark.parametrize("flags,M0,N0,K0", SIXTEEN_BIT)
def test_16_bit_operands(gpu_lib, flags, M0, N0, K0):  # noqa: F811
    for M, N, K, options in sixteen_bit_problems(M0, N0, K0):
        run_case(gpu_lib, flags, M, N, K, M0, N0, K0, "mmt4d_mfma_wave_tile", **options)


@pytest.mark.parametrize("M0,N0", FOUR_BIT)
def test_four_bit_rhs(gpu_lib, M0, N0):  # noqa: F811
    for M, N, K, options in four_bit_problems(M0, N0):
        run_case(gpu_lib, S8S4, M, N, K, M0, N0, 32, "mmt4d_mfma_wave_tile", **options)


# The k steps that chunk 0 shares with chunk 1 count once: an infinity there gives its row infinities and no NaN.
@pytest.mark.parametrize("rest", [1, 2, 3])
def test_an_infinity_in_what_two_chunks_share(gpu_lib, rest):  # noqa: F811
    M, N, K, K0 = 109, 132, 65 * 4 - rest, 8
    k = (4 - rest) * K0  # the first one
    lhs = torch.ones(M, K, 16, K0, dtype=torch.bfloat16, device="cuda")
    rhs = torch.ones(N, K, 16, K0, dtype=torch.bfloat16, device="cuda")
    lhs[3, k // K0, 5, 0] = float("inf")
    out = torch.zeros(M, N, 16, 16, device="cuda")
    p = mm_params(lhs.data_ptr(), rhs.data_ptr(), out.data_ptr(), M, N, K, 16, 16, K0, BF16)
    gpu_lib.iree_uk_mmt4d_p(C.byref(p))
    assert gpu_lib.iree_uk_mi355x_last_kernel() == b"mmt4d_mfma_wave_tile"
    want = torch.full((M, N, 16, 16), float(K * K0), device="cuda")
    want[3, :, 5, :] = float("inf")
    assert torch.equal(out, want)
