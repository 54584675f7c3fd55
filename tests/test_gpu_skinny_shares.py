"""The few-row kernel for narrow row pieces (mmt4d_skinny.hip) where its wavefronts' shares of the stream are empty, shorter
than the ring of loads, one ring, one and some; with streams that end inside a block of 1 KiB; for lhs tiles of 1, 2 and 4 rows
that are loaded a k step at a time, the same rows misaligned or in several tiles, which are not, and 8 rows; on both sides of
the lines at which the number of wavefronts and loads in flight changes (256 and 512 tile rows, 64, 96, 128 and 144 KiB a
tile, 48 and 128 MiB of rhs); every type and piece with streams that are longer than the ring.

Integers are compared bit for bit with a float64 product, floats within 1e-3 of max(|ref|, rms(ref)): sums of at most
8200 products of unit-scale values in 32 bits differ by about 1e-6 of that in any order.
"""
import pytest

from iree_amd import abi
from test_gpu_big_tiles import gpu_lib, run_case  # noqa: F401
from test_gpu_skinny_narrow import run_s16_case

pytestmark = pytest.mark.gpu

S8, F16, BF16, F32 = abi.MMT4D_TYPE_S8S8S32, abi.MMT4D_TYPE_F16F16F32, abi.MMT4D_TYPE_BF16BF16F32, abi.MMT4D_TYPE_F32F32F32
BYTES = {S8: 1, F16: 2, BF16: 2, F32: 4}


@pytest.mark.parametrize("flags,N0,K0", [(S8, 16, 2), (S8, 8, 4), (S8, 8, 8), (F16, 16, 1), (F16, 8, 4), (BF16, 16, 2), (BF16, 32, 1),
                                         (F32, 16, 1), (F32, 8, 2)])
@pytest.mark.parametrize("M,M0", [(1, 1), (1, 2), (1, 4), (2, 1), (3, 1), (2, 2)])
def test_shares(gpu_lib, flags, N0, K0, M, M0):  # noqa: F811
    g = K0 * BYTES[flags]
    per_kib = 1024 // (N0 * g)  # k steps in a block
    for n, blocks in enumerate([0, 1, 3, 4, 5, 8, 16, 17, 31, 32, 36, 60, 65, 100]):
        for K in {blocks * per_kib, blocks * per_kib + 1 + n % max(1, per_kib - 1)} - {0}:
            # (A misaligned lhs: one element in, or with K0 of 1 two; its pieces stay aligned.)
            offset = (K0 if n % 2 else 0)
            run_case(gpu_lib, flags, M, [16, 255, 257][n % 3], K, M0, N0, K0, "mmt4d_skinny", lhs_pad=K0 * (n % 2),
                     rhs_pad=16 // BYTES[flags] * (n % 2), out_pad=4 * (n % 2), offsets=(offset, 16 // BYTES[flags] * (n % 2), 0),
                     accumulate=n % 3 == 1, seed=n)


@pytest.mark.parametrize("flags,K0", [(S8, 2), (F16, 1), (BF16, 2), (F32, 2)])
@pytest.mark.parametrize("M0", [1, 2, 4])
def test_tile_sizes(gpu_lib, flags, K0, M0):  # noqa: F811
    kib = 1024 // (16 * K0 * BYTES[flags])
    for N, tile_kib in [(16, 256), (256, 64), (257, 63), (512, 20), (513, 63), (513, 64), (600, 95), (600, 96), (600, 100), (520, 127), (520, 128), (513, 143),
                        (513, 144), (200, 256)]:
        if N * tile_kib < 76 << 10:
            run_case(gpu_lib, flags, 1, N, tile_kib * kib, M0, 16, K0, "mmt4d_skinny", seed=N)


# int8 in pieces of one byte, two k steps a lane: the stream ends behind a lane's first k step or its second (rhs tile rows
# stay 16-byte multiples apart).
@pytest.mark.parametrize("M,M0", [(1, 1), (1, 2), (1, 4), (3, 1), (2, 4)])
def test_one_byte_pieces_long_streams(gpu_lib, M, M0):  # noqa: F811
    for n, (N, tile_kib) in enumerate([(16, 40), (256, 100), (257, 64), (513, 41), (600, 100)]):
        for K in (128 * tile_kib, 128 * tile_kib + 35):
            run_case(gpu_lib, S8, M, N, K, M0, 8, 1, "mmt4d_skinny", rhs_pad=8 * (K % 2), accumulate=n % 2 == 1, seed=n)


@pytest.mark.parametrize("M,M0,N0", [(1, 1, 16), (1, 2, 16), (1, 4, 16), (1, 8, 16), (3, 4, 16), (7, 1, 32)])
def test_int4_one_byte_pieces_long_streams(gpu_lib, M, M0, N0):  # noqa: F811
    for n, (N, tile_kib) in enumerate([(16, 40), (256, 64), (257, 100), (513, 41), (600, 100)]):
        K = tile_kib * 1024 // N0 + n
        run_case(gpu_lib, abi.MMT4D_TYPE_S8S4S32, M, N, K, M0, N0, 2, "mmt4d_skinny", accumulate=n % 2 == 1, seed=n)


# More than two tile rows a unit, from the caches and from HBM (one byte an element and several rows: above 128 MiB).
@pytest.mark.parametrize("M0", [1, 4, 8])
@pytest.mark.parametrize("kind,N0,K0,g", [("s16", 16, 2, 4), ("u4", 32, 8, 4), ("s8", 16, 2, 2), ("s8", 8, 8, 8)])
def test_sixteen_bit_integers_many_tile_rows(gpu_lib, kind, N0, K0, g, M0):  # noqa: F811
    for N, tile_kib in [(513, 21), (600, 100), (1040, 130)]:
        if N < 1000 or (kind != "s16" and M0 > 1):
            run_s16_case(gpu_lib, {"s16": False, "u4": True, "s8": "s8"}[kind], 1, N, tile_kib * 1024 // (N0 * g) + 1, M0, N0, K0,
                         N == 600, "mmt4d_skinny", seed=N)


@pytest.mark.parametrize("M0", [1, 4, 8])
@pytest.mark.parametrize("flags,N0,K0,g", [(abi.MMT4D_TYPE_S8S4S32, 16, 2, 1), (abi.MMT4D_TYPE_S8S4S32, 8, 8, 4), (S8, 16, 2, 2),
                                           (abi.MMT4D_TYPE_F16F16F16, 16, 1, 2), (abi.MMT4D_TYPE_BF16BF16BF16, 16, 2, 4)])
def test_other_types_many_tile_rows(gpu_lib, flags, N0, K0, g, M0):  # noqa: F811
    one_byte = flags in (S8, abi.MMT4D_TYPE_S8S4S32)
    M, M0 = (2, 4) if M0 == 8 and not flags == abi.MMT4D_TYPE_S8S4S32 else (1, M0)  # (8 rows a matrix kernel does not take)
    if M * M0 == 8 and flags == abi.MMT4D_TYPE_BF16BF16BF16:
        M, M0 = 8, 1
    for N, tile_kib in [(513, 21), (600, 100), (1040, 130)]:
        if N < 1000 or (one_byte and M * M0 > 1):
            run_case(gpu_lib, flags, M, N, tile_kib * 1024 // (N0 * g) + 1, M0, N0, K0, "mmt4d_skinny", accumulate=N == 600, seed=N)
