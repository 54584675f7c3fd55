"""The block kernels' loads that take 64 contiguous bytes per four lanes (mmt4d_mfma_kernels.h): 4-byte row pieces with tiles of
4, 8 and 16 rows in every combination of the operands, which share one order of k inside a chunk, and 64-byte row pieces and
one-row tiles, whose columns are exclusive-ored into place. K from one chunk to several, ending at every place of a chunk that
row pieces leave; ragged last tiles. Tolerances as in test_gpu_big_tiles: integers exact.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401

pytestmark = pytest.mark.gpu

S8, BF16, F32 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_BF16BF16F32, abi.MMT4D_TYPE_F32F32F32
# Rows and columns that 64x64, 128x64, 128x128, 192x192 and 256x256 tiles are taken for.
SIZES = [(72, 14000), (200, 4168), (1000, 2056), (2000, 4168), (3608, 3704)]


@pytest.mark.parametrize("flags,e", [(S8, 1), (BF16, 2), (F32, 4)])
@pytest.mark.parametrize("M0,N0", [(8, 8), (16, 8), (8, 16), (4, 8), (8, 4), (16, 4), (16, 16)])
def test_four_byte_pieces(gpu_lib, flags, e, M0, N0):  # noqa: F811
    for n, (rows, cols) in enumerate(SIZES):
        if flags == F32 and n not in (2, 4):
            continue
        # 16 k steps are a chunk: whole, and each remainder once over the sizes
        for K in (16, 17 + (3 * n + M0) % 15, 48 + (7 * n + N0) % 16):
            run_case(gpu_lib, flags, rows // M0, cols // N0, K, M0, N0, 4 // e, "mmt4d_mfma_*", out_pad=4 if n % 2 else 0,
                     accumulate=K > 32, seed=n)


@pytest.mark.parametrize("flags,e", [(S8, 1), (BF16, 2)])
@pytest.mark.parametrize("M0,N0,piece", [(16, 16, 64), (8, 8, 64), (4, 16, 64), (1, 16, 64), (1, 16, 32), (16, 4, 64)])
def test_rows_of_64_bytes(gpu_lib, flags, e, M0, N0, piece):  # noqa: F811
    for n, (rows, cols) in enumerate(SIZES):
        for K in (1, 3, 9, 16):
            run_case(gpu_lib, flags, rows // M0, cols // N0, K * (64 // piece) + (K % 2 if piece == 32 else 0), M0, N0, piece // e,
                     "mmt4d_mfma_*", lhs_pad=64 // e if K == 3 else 0, accumulate=K == 3, seed=n)
